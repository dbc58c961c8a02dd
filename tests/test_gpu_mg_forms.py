"""Multigrid kernels at the batch sizes where the form changes, and with windows up to the whole cube (needs an MI355X).

A batch repeats a few distinct patches; each copy must be bitwise the oracle's result at a fixed number of V-cycles (the
kernels keep the reference's operation order), whatever the batch size."""
import numpy as np
import pytest

import gpu_testbed_poisson_gravity_amd as pg
import oracle as O
from gpu_testbed_poisson_gravity_amd import inputs as I

pytestmark = pytest.mark.gpu
POI = 4.0 * np.pi * 1e-5
K = 7   # distinct patches


def _patches(gs, dtype):
    rho, cpot, flu, _ = I.plummer(K, gs, seed=60 + gs, dtype=dtype)
    flu[:, 1:4] = 0.05 * np.sin(np.arange(flu[:, 1:4].size)).reshape(flu[:, 1:4].shape)
    return rho, cpot, flu


def _check(gs, n, dtype, gg=1, init=pg.INIT_INTERP, graacc=True, guess=None, quad=False, smooth=(2, 3), p5=False):
    rho, cpot, flu = _patches(gs, dtype)
    at = np.arange(n) % K
    ints = pg.INT_QUAD if quad else pg.INT_CQUAD
    kw = dict(mg_max_iter=3, mg_npre=smooth[0], mg_npost=smooth[1], mg_tol=0.0, poi_coeff=POI, dt=0.5, dh=0.75, p5=p5)
    print(f"[case] mg gs={gs} n={n} {np.dtype(dtype).name} gg={gg} init={init} quad={quad} smooth={smooth} p5={p5}", flush=True)
    solve = pg.solve_host if dtype == np.float32 else pg.solve_host_f64
    pot, fl, it, st = solve(rho[at], cpot[at], flu[at] if graacc else None, gs=gs, gg=gg, scheme=pg.MG, init_mode=init,
                            guess=None if guess is None else guess[at], int_scheme=ints, graacc=graacc, **kw)
    p = O.make_params(gs=gs, gg=min(gg, 2), scheme=O.MG, init_mode=init, int_scheme=ints, graacc=graacc, **kw)
    o_pot, o_fl, _, _ = O.solve(rho, cpot, flu if graacc else None, p, guess=guess, dtype=dtype)
    w = gg - min(gg, 2)   # the oracle's window is at most 12^3: the middle of a wider one
    assert np.all(it == 3)
    assert np.array_equal(pot[:, w:pot.shape[1] - w, w:pot.shape[1] - w, w:pot.shape[1] - w], o_pot[at])
    if graacc:
        assert np.array_equal(fl, o_fl[at])
    return pot, rho, cpot


@pytest.mark.parametrize("gs, n, dtype", [(1, 1, np.float32), (1, 1024, np.float32), (1, 1025, np.float32),
                                          (2, 512, np.float32), (2, 513, np.float32), (1, 512, np.float64),
                                          (1, 513, np.float64), (2, 256, np.float64), (2, 257, np.float64),
                                          (2, 1025, np.float64), (3, 9, np.float32), (4, 9, np.float64)])
def test_mg_forms_bitwise(gs, n, dtype):
    _check(gs, n, dtype)


@pytest.mark.parametrize("gs, n", [(1, 1030), (2, 520), (2, 3), (3, 3), (4, 3), (5, 3)])
def test_mg_options_bitwise(gs, n):
    """Zero start and caller's guess, quadratic interpolation, no pre- or post-smoothing, 5-point gradient."""
    guess = np.random.default_rng(gs).standard_normal((K,) + (6 + 2 * gs,) * 3).astype(np.float32) * 1e-4
    gg = min(gs, 2)
    _check(gs, n, np.float32, init=pg.INIT_ZERO, quad=True, smooth=(0, 2), gg=gg, p5=gg == 2)
    _check(gs, n, np.float32, init=pg.INIT_GUESS, guess=guess, smooth=(1, 0))


@pytest.mark.parametrize("gs", [1, 2, 3, 4, 5])
def test_mg_whole_cube_window(gs):
    """A Poisson-only window of the whole cube: its Dirichlet layer, edges and corners included, is the interpolated
    coarse potential (an SOR solve of no iterations from the interpolated start writes exactly that cube)."""
    n = 1030 if gs <= 2 else 5
    pot, rho, cpot = _check(gs, n, np.float32, gg=gs, graacc=False)
    cube, _, _, _ = pg.solve_host(rho, cpot, None, gs=gs, gg=gs, scheme=pg.SOR, sor_min_iter=0, sor_max_iter=0,
                                  graacc=False, poi_coeff=POI)
    shell = np.ones(pot.shape[1:], bool)
    shell[1:-1, 1:-1, 1:-1] = False
    assert np.array_equal(pot[:, shell], cube[np.arange(n) % K][:, shell])


@pytest.mark.parametrize("gs, n, dtype", [(1, 1536, np.float32), (1, 1537, np.float32), (1, 768, np.float64),
                                          (1, 769, np.float64), (3, 256, np.float32), (3, 257, np.float32),
                                          (3, 256, np.float64), (3, 257, np.float64)])
def test_mg_forms_bitwise_at_their_limits(gs, n, dtype):
    _check(gs, n, dtype)
    _check(gs, n, dtype, gg=gs, graacc=False, smooth=(1, 0))
