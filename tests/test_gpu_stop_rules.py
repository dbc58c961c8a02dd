"""Where a patch stops must not depend on how many patches share its call (needs an MI355X): the kernels come in several forms,
chosen by the batch size, whose threads hold different cells, and every form has to decide alike.  Tolerances and inputs are
therefore put within a few units in the last place of a tie, where the order of a sum would show."""
import numpy as np
import pytest

import gpu_testbed_poisson_gravity_amd as pg
from gpu_testbed_poisson_gravity_amd import inputs as I

pytestmark = pytest.mark.gpu
POI = 4.0 * np.pi * 1e-5


class _Solver:
    """Device solves of one set of patches, repeated to any batch size; returns potentials, counts and statuses."""

    def __init__(self, gs, dtype, rho, cpot, n, guess=None, **opts):
        import torch

        self.torch, self.f64, self.n, self.k = torch, dtype == np.float64, n, len(rho)
        at = np.arange(n) % self.k
        dev = lambda a: torch.as_tensor(np.ascontiguousarray(a[at])).cuda()   # noqa: E731
        self.rho, self.cpot, self.guess = dev(rho), dev(cpot), None if guess is None else dev(guess)
        self.ctx = pg.Context(0)
        self.opts = dict(pot_ghost_size=gs, gra_ghost_size=opts.pop("gra_ghost_size", 1), fuse_gravity=0, **opts)
        G = 8 + 2 * self.opts["gra_ghost_size"]
        self.out = torch.zeros((n, G, G, G), device="cuda", dtype=self.rho.dtype)
        self.it, self.st = (torch.zeros(n, dtype=torch.int32, device="cuda") for _ in range(2))

    def __call__(self, opts=None, **args):
        self.ctx.set_options(**dict(self.opts, **(opts or {})))
        a = (pg.solver_args_f64 if self.f64 else pg.solver_args)(poi_coeff=POI, graacc=False, **args)
        solve = self.ctx.solve_device_f64 if self.f64 else self.ctx.solve_device
        solve(self.rho, self.cpot, self.out, None, self.n, a, guess=self.guess, iters=self.it, status=self.st)
        self.torch.cuda.synchronize()
        return [x.cpu().numpy() for x in (self.out, self.it, self.st)]


def _around(x, dtype, ulps=12):
    """x and the `ulps` numbers of the type on either side of it."""
    x = dtype(x)
    return [dtype(x + i * np.spacing(x)) for i in range(-ulps, ulps + 1)]


def _agree(res, k):
    """Every copy of a patch, in every batch, has the same result."""
    ref = [x[:k] for x in res[0]]
    for r in res:
        for x, y in zip(r, ref):
            assert np.array_equal(x, y[np.arange(len(x)) % k])
    return ref


def _mg_error(rho, cube, dtype):
    """The multigrid error estimate of whole cubes at cell size 1: each cell's terms as the kernel forms them, exact sums."""
    c = cube[:, 1:-1, 1:-1, 1:-1]
    nb = cube[:, 2:, 1:-1, 1:-1] + cube[:, :-2, 1:-1, 1:-1] + cube[:, 1:-1, 2:, 1:-1] + cube[:, 1:-1, :-2, 1:-1]
    nb = nb + cube[:, 1:-1, 1:-1, 2:] + cube[:, 1:-1, 1:-1, :-2]
    d = dtype(-1) * (nb - dtype(6) * c) + dtype(POI) * rho
    s = [np.abs(x).astype(np.longdouble).sum(axis=(1, 2, 3)) for x in (d, c)]
    return s[0] / s[1]


@pytest.mark.parametrize("gs, sizes, dtype", [(1, (3, 1024, 1025), np.float32), (2, (3, 512, 513), np.float32),
                                              (1, (3, 512, 513), np.float64), (2, (3, 256, 257), np.float64),
                                              (1, (3, 1536, 1537), np.float32), (1, (3, 768, 769), np.float64),
                                              (3, (3, 256, 257), np.float32), (3, (3, 256, 257), np.float64)])
def test_mg_stops_alike_in_every_batch(gs, sizes, dtype):
    """Batch sizes on both sides of the line between one cell per thread and blocks of cells."""
    k = 3
    rho, cpot, _, _ = I.plummer(k, gs, seed=40 + gs, dtype=dtype)
    whole = _Solver(gs, dtype, rho, cpot, k, pot_scheme=pg.MG, gra_ghost_size=gs)
    runs = [_Solver(gs, dtype, rho, cpot, n, pot_scheme=pg.MG) for n in sizes]
    counts = set()
    for cycles in (1, 2):
        cube = whole(mg_max_iter=cycles, mg_tol=0.0)[0]
        for p, e in enumerate(_mg_error(rho, cube, dtype)):
            print(f"[case] mg gs={gs} {dtype.__name__} n={sizes} tolerances around patch {p}'s error {float(e):.4g}", flush=True)
            for tol in _around(e, dtype):
                counts.update(_agree([r(mg_max_iter=4, mg_tol=float(tol)) for r in runs], k)[1].tolist())
    assert {1, 2, 3} <= counts


@pytest.mark.parametrize("gs, sizes", [(1, (5, 1025, 1536, 1537)), (2, (5, 512, 513)), (3, (5, 256, 257))])
def test_mg_checks_guesses_alike_in_every_batch(gs, sizes):
    k, R, dtype = 5, 6 + 2 * gs, np.float32
    rho, cpot, _, _ = I.plummer(k, gs, seed=50 + gs)
    guess = (np.random.default_rng(gs).standard_normal((k, R, R, R)) * 1e-3).astype(np.float32)
    N = R + 2
    cube = _Solver(gs, dtype, rho, cpot, k, pot_scheme=pg.SOR, gra_ghost_size=gs)(sor_min_iter=0, sor_max_iter=0)[0]
    cube[:, 1:-1, 1:-1, 1:-1] = guess   # with the interpolated Dirichlet layer
    assert cube.shape == (k, N, N, N)
    c = cube[:, 1:-1, 1:-1, 1:-1]
    r = cube[:, 2:, 1:-1, 1:-1] + cube[:, :-2, 1:-1, 1:-1] + cube[:, 1:-1, 2:, 1:-1] + cube[:, 1:-1, :-2, 1:-1]
    r = r + cube[:, 1:-1, 1:-1, 2:] + cube[:, 1:-1, 1:-1, :-2] - dtype(6) * c - dtype(POI) * rho
    ratio = np.abs(r).sum(axis=(1, 2, 3), dtype=np.float64) / np.abs(c).sum(axis=(1, 2, 3), dtype=np.float64)
    runs = [_Solver(gs, dtype, rho, cpot, n, guess=guess, pot_scheme=pg.MG, init_mode=pg.INIT_GUESS) for n in sizes]
    fell = set()
    for p in range(k):
        print(f"[case] mg guess check gs={gs} n={sizes} tolerances around {ratio[p]:.4g}", flush=True)
        for tol in _around(ratio[p], dtype):
            res = [s(opts=dict(guess_fallback_tol=float(tol)), mg_max_iter=1, mg_tol=0.0) for s in runs]
            fell.add(bool(_agree(res, k)[2][p] & pg.STATUS_FALLBACK))
    assert fell == {False, True}


def test_mg_slices_and_mixed_modes_stop_alike():
    """A host batch cut into slices against the same batch in one launch, and both modes of a mixed batch."""
    import torch

    k, n, dtype = 3, 2056, np.float32   # slices of 1024, 512 and 520 patches, one launch of 2056
    at = np.arange(n) % k
    rho, cpot, _, _ = I.plummer(k, 1, seed=41)
    cube = _Solver(1, dtype, rho, cpot, k, pot_scheme=pg.MG, gra_ghost_size=1)(mg_max_iter=2, mg_tol=0.0)[0]
    one = _Solver(1, dtype, rho, cpot, n, pot_scheme=pg.MG)
    with pg.Context(0) as host, pg.Context(0) as mixed:
        host.set_options(pot_ghost_size=1, pot_scheme=pg.MG)
        h_rho, h_cpot, h_out, h_flu = host.mem_allocate(n // 8)
        h_rho[...], h_cpot[...] = rho[at], cpot[at]
        plan = mixed.plan(np.ones(n, np.int32), np.full(n, pg.MG, np.int32))
        small = mixed.plan(np.ones(k, np.int32), np.full(k, pg.MG, np.int32))
        d_rho, d_cpot = one.rho.reshape(-1), one.cpot.reshape(-1)
        d_out = torch.zeros_like(one.out)
        d_it, d_st = torch.zeros_like(one.it), torch.zeros_like(one.st)
        for tol in sum((_around(e, dtype) for e in _mg_error(rho, cube, dtype)), []):
            print(f"[case] mg gs=1 slices and mixed modes, tolerance {tol:.9g}", flush=True)
            kw = dict(mg_max_iter=4, mg_tol=float(tol))
            res = [one(**kw)]
            host.asyn_poisson_gravity_solver(h_rho, h_cpot, h_out, h_flu, n // 8, 1e-3, 1.0, 10, 10, 1.7, 4, 3, 3, float(tol),
                                             POI, pg.INT_CQUAD, False, True, False, gpu_nstream=1)
            host.synchronize()
            res.append([h_out.copy(), *host.patch_stats(n)])
            for persistent in (0, 1):
                mixed.set_options(mixed_persistent=persistent)
                for pl, m in ((plan, n), (small, k)):
                    mixed.solve_mixed_device(pl, d_rho, d_cpot, d_out, None, pg.solver_args(poi_coeff=POI, graacc=False, **kw),
                                             iters=d_it, status=d_st)
                    torch.cuda.synchronize()
                    res.append([x[:m].cpu().numpy() for x in (d_out, d_it, d_st)])
            _agree(res, k)
        plan.close()
        small.close()


def _bisect(changes, lo, hi, steps=56):
    """Neighbouring doubles: the last on lo's side for which changes(x) (an array) is false, with changes(hi) true."""
    lo, hi = np.array(lo, np.float64), np.array(hi, np.float64)
    assert not changes(lo).any() and changes(hi).all()
    for _ in range(steps):
        mid = lo + (hi - lo) / 2
        c = changes(mid)
        lo, hi = np.where(c, lo, mid), np.where(c, mid, hi)
    assert np.all(hi - lo <= 2 * np.spacing(lo))
    return lo


ULPS = np.arange(-24, 25)
FP64_SIZES = (512, 513, 700)   # ghost size 3: two planes per thread up to 512 patches, then four


@pytest.mark.parametrize("rule, tol", [(pg.TERM_RELRES, 2.0), (pg.TERM_RELRES, 1.0), (pg.TERM_RELRES, 0.5),
                                       (pg.TERM_REFERENCE, 0.0)])
def test_fp64_sor_stops_alike_in_every_batch(rule, tol):
    """The relaxation factor, the one double-precision setting of the rules, is put where a patch's count changes: in the
    first iterations, while the residuals are far above round-off, so that a step of one unit in the last place moves the
    sums by as little."""
    gs, k = 3, 6
    rho, cpot, _, _ = I.plummer(k, gs, seed=70, dtype=np.float64)
    if rule == pg.TERM_RELRES:   # 2 to 4 iterations at a factor of 1, more below
        opts, args, ends = dict(term_mode=rule, rel_tol=tol, init_mode=pg.INIT_ZERO), dict(sor_min_iter=0, sor_max_iter=20), (0.6, 1.0)
    else:                        # the residual grows after two or three iterations above a factor of about 1.9
        opts, args, ends = dict(term_mode=rule), dict(sor_min_iter=0, sor_max_iter=20), (1.6, 1.9)
    few = _Solver(gs, np.float64, rho, cpot, k, **opts)
    runs = [few] + [_Solver(gs, np.float64, rho, cpot, n, **opts) for n in FP64_SIZES]
    most = few(sor_omega=ends[1], **args)[1]
    for p in range(k):
        at = _bisect(lambda w: few(sor_omega=float(w), **args)[1][p] <= most[p], *ends)
        print(f"[case] f64 gs=3 rule {rule}: patch {p}, factors around {float(at):.6f}", flush=True)
        got = {int(_agree([r(sor_omega=float(at + u * np.spacing(at)), **args) for r in runs], k)[1][p]) for u in ULPS}
        assert len(got) > 1


def test_fp64_sor_checks_guesses_alike_in_every_batch():
    """The solution of a density as the guess, and the density scaled to where the guess fails (its tolerance is in single
    precision)."""
    gs, k, N = 3, 8, 14
    rho, cpot, _, _ = I.plummer(k, gs, seed=70, dtype=np.float64)
    cube = _Solver(gs, np.float64, rho, cpot, k, term_mode=pg.TERM_RELRES, gra_ghost_size=gs)(
        sor_min_iter=10, sor_max_iter=400, sor_omega=1.6)[0]
    assert cube.shape == (k, N, N, N)
    guess = np.ascontiguousarray(cube[:, 1:-1, 1:-1, 1:-1])
    ratio = np.abs(POI * rho).sum(axis=(1, 2, 3)) / np.abs(guess).sum(axis=(1, 2, 3))
    opts = dict(term_mode=pg.TERM_RELRES, init_mode=pg.INIT_GUESS, guess_fallback_tol=float(ratio.max()))
    args = dict(sor_min_iter=0, sor_max_iter=0)
    few = _Solver(gs, np.float64, rho, cpot, k, guess=guess, **opts)

    def fails(s):
        few.rho.copy_(few.torch.as_tensor(rho * s[:, None, None, None]))
        return (few(**args)[2] & pg.STATUS_FALLBACK) != 0

    at = _bisect(fails, np.ones(k), np.full(k, 2 + ratio.max() / ratio.min()))
    s = (at[:, None] + ULPS * np.spacing(at)[:, None]).reshape(-1)
    pick = np.repeat(np.arange(k), ULPS.size)
    many = rho[pick] * s[:, None, None, None], cpot[pick]
    print(f"[case] f64 gs=3 guess check: {s.size} scales", flush=True)
    res = [_Solver(gs, np.float64, *many, n, guess=guess[pick], **opts)(**args) for n in (s.size,) + FP64_SIZES]
    fell = (_agree(res, s.size)[2] & pg.STATUS_FALLBACK).reshape(k, -1) != 0
    assert np.all(fell.any(axis=1) & ~fell.all(axis=1))
