"""Large one-stream batches from host arrays run in slices (needs an MI355X): they must return what the plain sequence
returns, which a call with two streams takes, bit for bit, with pinned and pageable arrays, for calls that follow each other
without a synchronize, and with arrays that overlap."""
import numpy as np
import pytest

import gpu_testbed_poisson_gravity_amd as pg
from gpu_testbed_poisson_gravity_amd import inputs as I

pytestmark = pytest.mark.gpu
POI = 4.0 * np.pi * 1e-5


def _inputs(n, gs):
    rho, cpot, flu, _ = I.plummer(64, gs, seed=7 * gs)
    k = np.arange(n) % 61
    scale = (1.0 + np.arange(n) / n).astype(np.float32)[:, None, None, None]
    return rho[k] * scale, cpot[k] * scale, flu[k].copy()


def _call(ctx, arrays, n, streams, scheme, poisson=True, graacc=True):
    it = (3, 3, 1.0) if scheme == pg.MG else (10, 60, 1.7)
    ctx.asyn_poisson_gravity_solver(*arrays, n // 8, 1e-3, 1.0, *it, 4, 2, 2, 1e-6, POI, pg.INT_CQUAD, False, poisson,
                                    graacc, gpu_nstream=streams)


@pytest.mark.parametrize("pinned", [True, False])
@pytest.mark.parametrize("gs, scheme, n, poisson, graacc", [(5, pg.SOR, 1024, True, True), (2, pg.SOR, 1016, True, True),
                                                            (1, pg.SOR, 2056, True, False), (3, pg.MG, 1544, True, True),
                                                            (1, pg.SOR, 1032, False, True)])
def test_slices_match_the_sequence(gs, scheme, n, poisson, graacc, pinned):
    rho, cpot, flu = _inputs(n, gs)
    res = {}
    for streams in (2, 1):
        print(f"[case] host gs={gs} scheme={scheme} n={n} streams={streams} pinned={pinned}", flush=True)
        with pg.Context(0) as ctx:
            ctx.set_options(pot_ghost_size=gs, gra_ghost_size=1, pot_scheme=scheme)
            arrays = ctx.mem_allocate(n // 8)
            if not pinned:
                arrays = [np.zeros_like(a) for a in arrays]
            for a, x in zip((arrays[0], arrays[1], arrays[3]), (rho, cpot, flu)):
                a[...] = x
            arrays[2][...] = 0.25 * np.cos(np.arange(arrays[2].size)).reshape(arrays[2].shape)
            for m in (n, n - 8):   # the second call has other slices and reads the fluid that the first one wrote
                _call(ctx, arrays, m, streams, scheme, poisson, graacc)
                if not pinned:
                    ctx.synchronize()
            ctx.synchronize()
            res[streams] = [a.copy() for a in arrays[2:]] + (list(ctx.patch_stats(n - 8)) if poisson else [])
    for x, y in zip(res[1], res[2]):
        assert np.array_equal(x, y)


def test_overlapping_arrays_keep_the_sequence():
    n, gs = 1024, 1
    rho, cpot, flu = _inputs(n, gs)
    res = []
    for streams in (2, 1):
        print(f"[case] host overlap streams={streams}", flush=True)
        with pg.Context(0) as ctx:
            ctx.set_options(pot_ghost_size=gs, gra_ghost_size=1)
            h_rho, h_cpot, h_out, h_flu = ctx.mem_allocate(n // 8)
            h_rho[...], h_cpot[...], h_flu[...] = rho, cpot, flu
            # the potential [n][10^3] goes over the density [n][R^3] and the coarse cubes, which it is larger than
            both = np.zeros(max(h_out.size, h_rho.size), np.float32)
            both[:h_rho.size] = h_rho.ravel()
            _call(ctx, (both[:h_rho.size].reshape(h_rho.shape), h_cpot, both[:h_out.size].reshape(h_out.shape), h_flu), n,
                  streams, pg.SOR)
            ctx.synchronize()
            res.append((both[:h_out.size].copy(), h_flu.copy()))
    for x, y in zip(*res):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("pinned", [True, False])
@pytest.mark.parametrize("gs, n, poisson", [(1, 1528, False), (2, 1544, False), (2, 2056, True), (4, 4104, True)])
def test_slices_match_at_their_limits(gs, n, poisson, pinned):
    """Gravity alone around its smallest sliced batch, and batches of several slices that pageable arrays get two of; the
    test's second call of each is 8 patches smaller."""
    test_slices_match_the_sequence(gs, pg.SOR, n, poisson, True, pinned)
