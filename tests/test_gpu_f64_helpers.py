"""FP64 SOR at ghost size 1, where batches of up to 1536 patches run with three waves beside the one that has a patch's cells
(needs an MI355X): bit for bit the FP64 oracle's results, and the same results and counts on both sides of that size."""
import numpy as np
import pytest

import gpu_testbed_poisson_gravity_amd as pg
import oracle as O
from gpu_testbed_poisson_gravity_amd import inputs as I
from test_gpu_f64 import POI

pytestmark = pytest.mark.gpu
K, R, N = 6, 8, 10
SIZES = (K, 1536, 1537)


def _patches():
    rho, cpot, flu, _ = I.plummer(K, 1, seed=33, dtype=np.float64)
    flu[:, 1:4] = 0.05 * np.sin(np.arange(flu[:, 1:4].size)).reshape(flu[:, 1:4].shape)
    return rho, cpot, flu


def _solve(n, rho, cpot, flu, guess=None, guess_tol=0.0, rel_tol=1e-5, **kw):
    import torch

    at = np.arange(n) % K
    dev = lambda a: None if a is None else torch.as_tensor(np.ascontiguousarray(a[at])).cuda()   # noqa: E731
    opts = {k: kw.pop(k) for k in ("init_mode", "term_mode", "check_every", "fuse_gravity") if k in kw}
    with pg.Context(0) as ctx:
        ctx.set_options(pot_ghost_size=1, gra_ghost_size=1, rel_tol=rel_tol, guess_fallback_tol=guess_tol, **opts)
        out, d_flu = torch.zeros((n, N, N, N), dtype=torch.float64, device="cuda"), dev(flu)
        it, st = (torch.zeros(n, dtype=torch.int32, device="cuda") for _ in range(2))
        ctx.solve_device_f64(dev(rho), dev(cpot), out, d_flu, n, pg.solver_args_f64(poi_coeff=POI, dt=0.5, **kw),
                             guess=dev(guess), iters=it, status=st)
        torch.cuda.synchronize()
    return [x.cpu().numpy() for x in (out, d_flu, it, st)]


def _all_sizes(*a, **kw):
    ref = _solve(K, *a, **kw)
    for n in SIZES[1:]:
        for x, y in zip(_solve(n, *a, **kw), ref):
            assert np.array_equal(x, y[np.arange(n) % K], equal_nan=x.dtype.kind == "f")
    return ref


@pytest.mark.parametrize("quad", [False, True])
@pytest.mark.parametrize("init", [pg.INIT_INTERP, pg.INIT_ZERO, pg.INIT_GUESS])
@pytest.mark.parametrize("iters", [0, 1, 7])
def test_helpers_match_oracle(init, iters, quad):
    x = _patches()
    guess = np.cos(np.arange(K * R ** 3, dtype=np.float64)).reshape(K, R, R, R) if init == pg.INIT_GUESS else None
    kw = dict(sor_min_iter=iters, sor_max_iter=iters, sor_omega=1.49, int_scheme=pg.INT_QUAD if quad else pg.INT_CQUAD)
    print(f"[case] f64 gs=1 helpers init={init} iters={iters} quad={quad}", flush=True)
    pot, flu, it, _ = _all_sizes(*x, guess=guess, init_mode=init, **kw)
    o = O.solve(*x, O.make_params(gs=1, gg=1, init_mode=init, poi_coeff=POI, dt=0.5, **kw), guess=guess, dtype=np.float64)
    assert np.array_equal(pot, o[0]) and np.array_equal(flu, o[1]) and np.array_equal(it, o[2])


def test_helpers_keep_rules_guesses_and_flags():
    rho, cpot, flu = _patches()
    print("[case] f64 gs=1 helpers: rules, whole-cube guesses, non-finite values", flush=True)
    kw = dict(sor_min_iter=10, sor_max_iter=200, sor_omega=1.49)
    it = _all_sizes(rho, cpot, flu, term_mode=pg.TERM_REFERENCE, **kw)[2]
    assert it.max() < 200
    for every in (1, 3):
        st = _all_sizes(rho, cpot, flu, term_mode=pg.TERM_RELRES, check_every=every, fuse_gravity=0, **kw)[3]
        assert np.all(st == pg.STATUS_CONVERGED)
    cube = _solve(K, rho, cpot, flu, term_mode=pg.TERM_RELRES, **kw)[0]
    cube[::2, 1:-1, 1:-1, 1:-1] *= 3.0
    st = _all_sizes(rho, cpot, flu, guess=cube, guess_tol=1e-2, init_mode=pg.INIT_GUESS_CUBE, term_mode=pg.TERM_RELRES, **kw)[3]
    assert np.array_equal((st & pg.STATUS_FALLBACK) != 0, np.arange(K) % 2 == 0)
    rho[2, 1, 2, 3], cpot[4, 0, 0, 0] = np.nan, np.inf
    st = _all_sizes(rho, cpot, flu, term_mode=pg.TERM_RELRES, **kw)[3]
    # a coarse corner reaches the cube's corner alone, which no stencil reads and which the flag does not cover
    assert np.array_equal((st & pg.STATUS_NONFINITE) != 0, np.arange(K) == 2)


def test_smallest_patches_are_not_the_slowest():
    """Ten iterations of 8 patches: fewer cells must not take longer than ghost size 2's."""
    import torch

    best = {}
    for gs in (1, 2):
        rho, cpot, _, _ = I.plummer(8, gs, seed=1, dtype=np.float64)
        rho, cpot = torch.as_tensor(rho).cuda(), torch.as_tensor(cpot).cuda()
        out = torch.zeros((8, N, N, N), dtype=torch.float64, device="cuda")
        args = pg.solver_args_f64(sor_min_iter=10, sor_max_iter=10, poi_coeff=POI, graacc=False)
        s = torch.cuda.current_stream().cuda_stream
        with pg.Context(0) as ctx:
            ctx.set_options(pot_ghost_size=gs, fuse_gravity=0)
            best[gs] = 1e9
            for _ in range(10):
                e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
                e[0].record()
                for _ in range(50):
                    ctx.solve_device_f64(rho, cpot, out, None, 8, args, stream=s)
                e[1].record()
                torch.cuda.synchronize()
                best[gs] = min(best[gs], e[0].elapsed_time(e[1]) / 50)
    print(f"[case] f64 8 patches, 10 iterations: gs=1 {best[1]:.4f} ms, gs=2 {best[2]:.4f} ms", flush=True)
    assert best[1] < 1.1 * best[2]
