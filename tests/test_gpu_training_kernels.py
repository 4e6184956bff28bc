"""Closure training kernels at the edges of their shapes: the gradient of 64-sample workgroups with full,
ragged and single-sample batches, and the summing of few and many partials, against float64 autograd."""

from __future__ import annotations

import pytest
import torch

from tensorlbm_amd import closure as cl

pytestmark = pytest.mark.gpu


def _case(n, seed):
    g = torch.Generator().manual_seed(seed)
    x = 4e-3 * torch.randn(n, 7, generator=g)
    t = 1e-3 * torch.rand(n, generator=g)
    model = cl.EddyViscosityMLP3D("cuda:0", seed=seed)
    model.set_feature_stats(1e-4 * torch.randn(7, generator=g), 3e-3 + 1e-3 * torch.rand(7, generator=g))
    return model, x, t


def _split(vec):
    p = vec.detach().double().cpu()
    return [p[:224].reshape(32, 7), p[224:256], p[256:1280].reshape(32, 32), p[1280:1312], p[1312:1344], p[1344:1345],
            p[1345:1352], p[1352:1359]]


def _reference(vec, x, t):
    w = [a.clone().requires_grad_(i < 6) for i, a in enumerate(_split(vec))]
    h = torch.relu((x.double() - w[6]) * w[7] @ w[0].T + w[1])
    z = torch.relu(h @ w[2].T + w[3]) @ w[4] + w[5]
    loss = ((torch.nn.functional.softplus(10 * z, threshold=1e9) / 10 - t.double()) ** 2).mean()
    loss.backward()
    return loss.item(), torch.cat([a.grad.reshape(-1) for a in w[:6]])


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 128, 129, 200, 4096, 4097])
def test_gradient_matches_autograd(n):
    model, x, t = _case(n, n)
    loss, grad = cl.mlp_loss_and_grad(model, x.to("cuda:0"), t.to("cuda:0"))
    want_loss, want = _reference(model.params, x, t)
    # fp32 sums of at most 64 terms per partial and n / 64 partials; units at a ReLU edge may flip, none do
    assert abs(float(loss) - want_loss) <= 2e-5 * want_loss
    assert float((grad.double().cpu() - want).abs().max()) <= 2e-5 * float(want.abs().max())


@pytest.mark.parametrize("n", [1, 64, 77, 256, 1000])
def test_predict_matches_float64(n):
    model, x, _ = _case(n, 7 * n)
    w = _split(model.params)
    h = torch.relu((x.double() - w[6]) * w[7] @ w[0].T + w[1])
    z = torch.relu(h @ w[2].T + w[3]) @ w[4] + w[5]
    want = torch.nn.functional.softplus(10 * z, threshold=1e9) / 10
    got = model(x.to("cuda:0")).reshape(-1).double().cpu()
    # softplus at slope <= 1 of a sum of 32 products of O(1): a few ulp of fp32 on z
    assert float((got - want).abs().max()) <= 4e-6


@pytest.mark.parametrize("n,batch", [(1, 8), (64, 64), (130, 64), (1000, 96), (1000, 1000), (333, 1)])
def test_epoch_matches_single_steps(n, batch):
    """The epoch's gathered rows, last short minibatch, step numbers and loss sum, against one step at a time.

    Both sum the same partials, in another order: parameters differ by rounding (Adam's step is at most lr
    per parameter, so a relative difference of 1e-4 in a gradient near zero moves one by 1e-4 lr)."""
    a, x, t = _case(n, 3 * n + batch)
    b = cl.clone_model(a)
    x, t = x.to("cuda:0"), t.to("cuda:0")
    order = torch.randperm(n, generator=torch.Generator().manual_seed(n)).to("cuda:0")
    oa, ob = (cl._Adam(m, 1e-3, max_batch=batch) for m in (a, b))
    want, steps = 0.0, 0
    for s in range(0, n, batch):
        idx = order[s:s + batch]
        want += float(oa.step(x[idx].contiguous(), t[idx].contiguous())[0].double()) * idx.shape[0]
        steps += 1
    got = float(ob.epoch(x, t, order, batch))
    assert oa.t == ob.t == steps
    assert abs(got - want) <= 1e-5 * abs(want)
    assert float((a.params - b.params).abs().max()) <= 1e-3 * 1e-3 * steps
    assert float((oa.m - ob.m).abs().max()) <= 1e-4 * float(oa.m.abs().max())


def test_epoch_refuses_bad_arguments():
    from tensorlbm_amd import _native as nat

    lib = nat.lib()
    ok = (4096,) * 4
    tail = (4096, 4096, 4096)
    rates = (1e-3, 0.9, 0.999, 1e-8, 1.0)
    assert lib.tlbm_mlp_train_epoch(*ok, 0, 8, *tail, 1, *rates, 4096, None) == nat.ERR_SHAPE
    assert lib.tlbm_mlp_train_epoch(*ok, 8, 0, *tail, 1, *rates, 4096, None) == nat.ERR_SHAPE
    assert lib.tlbm_mlp_train_epoch(*ok, 8, 8, *tail, 0, *rates, 4096, None) == nat.ERR_INVALID
    assert lib.tlbm_mlp_train_epoch(*ok, 8, 8, *tail, 1, *rates, None, None) == nat.ERR_INVALID
