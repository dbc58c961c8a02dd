"""FP64 SOR at ghost size 5, whose cube holds the cells of a column in pairs (needs an MI355X): every start, output
windows up to the whole cube, and counts down to one iteration, bit for bit those of the FP64 oracle."""
import numpy as np
import pytest

import gpu_testbed_poisson_gravity_amd as pg
import oracle as O
from test_gpu_f64 import OMEGA, POI, _inputs

pytestmark = pytest.mark.gpu
N = 5


def _solve(rho, cpot, flu, gg, init, iters, guess):
    kw = dict(dt=0.5, sor_min_iter=iters, sor_max_iter=iters, sor_omega=OMEGA[4], poi_coeff=POI)
    grav = gg <= 2   # wider windows are Poisson-only
    print(f"[case] f64 gs=5 gg={gg} init={init} iters={iters}", flush=True)
    return pg.solve_host_f64(rho, cpot, flu if grav else None, gs=5, gg=gg, init_mode=init, guess=guess, graacc=grav, **kw)


def _oracle(rho, cpot, flu, gg, init, iters, guess):
    p = O.make_params(gs=5, gg=gg, init_mode=init, sor_min_iter=iters, sor_max_iter=iters, sor_omega=OMEGA[4],
                      poi_coeff=POI, dt=0.5)
    return O.solve(rho, cpot, flu, p, guess=guess, dtype=np.float64)


def _guess():
    return np.cos(np.arange(N * 16 ** 3, dtype=np.float64)).reshape(N, 16, 16, 16)


@pytest.mark.parametrize("iters", [1, 6])
@pytest.mark.parametrize("init", [pg.INIT_INTERP, pg.INIT_ZERO, pg.INIT_GUESS])
@pytest.mark.parametrize("gg", [1, 2, 5])
def test_pairs_match_oracle(gg, init, iters):
    x, rest = _inputs(N, 5, seed=300 + gg), (init, iters, _guess() if init == pg.INIT_GUESS else None)
    g, o = _solve(*x, gg, *rest), _oracle(*x, min(gg, 2), *rest)
    k = gg - min(gg, 2)   # the whole cube holds the oracle's widest window
    assert np.array_equal(g[0][:, k:, k:, k:][:, :o[0].shape[1], :o[0].shape[1], :o[0].shape[1]], o[0])
    assert np.array_equal(g[2], o[2])
    assert gg > 2 or np.array_equal(g[1], o[1])


def test_whole_cube_guess_matches_interior_guess():
    """The guess as the whole cube, its Dirichlet layer taken from the whole-cube window of the other solve."""
    x = _inputs(N, 5, seed=310)
    a = _solve(*x, 5, pg.INIT_GUESS, 4, _guess())
    cube = a[0].copy()
    cube[:, 1:-1, 1:-1, 1:-1] = _guess()
    b = _solve(*x, 5, pg.INIT_GUESS_CUBE, 4, cube)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[2], b[2])
