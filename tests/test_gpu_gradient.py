"""Gradient sums of the warm-start network at the batch sizes where the split changes (needs an MI355X): one partial
per sample up to 128 samples, then several samples per partial with a remainder."""
import numpy as np
import pytest

import gpu_testbed_poisson_gravity_amd as pg
from oracle import cnn_oracle as CO
from test_gpu_cnn import TOL_GRAD, _dev, _random_params, _random_x0, _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, res_weight", [(1, 1.0), (17, 0.0), (130, 1.0)])
def test_gradient_sums_match_oracle(n, res_weight):
    import torch

    p = _random_params(20 + n)
    bits, x0 = _random_x0(n, seed=n)   # values in the border voxels too
    tgt = np.random.default_rng(n).normal(0, 0.5, (n, 512, 8)).astype(np.float32)
    with pg.Context(0) as ctx:
        net = pg.CNN(ctx)
        net.set_params(p)
        net.set_loss(res_weight)
        d_g = torch.empty(CO.NPARAMS, device="cuda")
        print(f"[case] loss_grad n={n} res_weight={res_weight}", flush=True)
        loss = net.loss_grad(_dev(bits.view(np.int16)), _dev(tgt), n, d_g)
        torch.cuda.synchronize()
        g = d_g.cpu().numpy()
        net.close()
    loss_o, g_o = CO.loss_grad(p, x0, tgt, bf16=True, res_weight=res_weight)
    assert abs(loss - loss_o) <= 1e-4 * loss_o
    for l in range(1, 7):
        for o, ln in ((CO.OW[l], 16 * 432), (CO.OB[l], 16)):
            assert _rel(g[o:o + ln], g_o[o:o + ln]) < TOL_GRAD, (l, ln)


@pytest.mark.parametrize("res_weight", [0.0, 1.0])
def test_several_samples_per_workgroup(res_weight):
    """More samples than workgroups, a remainder, border values in the packed input and a target at 4-byte alignment."""
    import torch

    n = 259
    p = _random_params(7)
    bits, x0 = _random_x0(n, seed=n)
    tgt = np.random.default_rng(n).normal(0, 0.5, (n, 512, 8)).astype(np.float32)
    buf = torch.empty(tgt.size + 1, device="cuda")
    buf[1:] = _dev(tgt).reshape(-1)
    with pg.Context(0) as ctx:
        net = pg.CNN(ctx)
        net.set_params(p)
        net.set_loss(res_weight)
        d_g = torch.empty(CO.NPARAMS, device="cuda")
        print(f"[case] loss_grad n={n} res_weight={res_weight}", flush=True)
        loss = net.loss_grad(_dev(bits.view(np.int16)), buf[1:], n, d_g)
        torch.cuda.synchronize()
        g = d_g.cpu().numpy()
        net.close()
    loss_o, g_o = CO.loss_grad(p, x0, tgt, bf16=True, res_weight=res_weight)
    assert abs(loss - loss_o) <= 1e-4 * loss_o
    for l in range(1, 7):
        for o, ln in ((CO.OW[l], 16 * 432), (CO.OB[l], 16)):
            assert _rel(g[o:o + ln], g_o[o:o + ln]) < TOL_GRAD, (l, ln)
