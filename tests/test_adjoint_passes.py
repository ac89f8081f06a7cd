"""A trajectory's gradient belongs to its own forward pass: with other passes of
the same engine, complete or failed, between a forward and its backward pass.
The library keeps one trajectory, so the autograd function runs its own again."""
import numpy as np
import pytest
import torch

import gamdpy_amd as gp
from gamdpy_amd import adjoint
from helpers import KA_EPS, KA_SIG


class OneTrajectory:
    """Stands in for an AdjointEngine: H = sigma^2 per class, and only the
    last forward pass can be differentiated."""
    ntypes, passes, last = 1, 0, None

    def forward(self, params, r0, v0):
        self.passes += 1
        self.last = None
        if params[0, 0, 0] <= 0:
            raise gp._native.NativeError("sigma")
        self.last = np.array(params[0, 0, 0], np.float64), np.array(r0), np.array(v0)
        return np.full((1, 1), self.last[0] ** 2)

    def backward(self, g):
        s, r0, v0 = self.last
        return np.array([[2 * s * g[0, 0], 0.0]]), g[0, 0] * r0, v0


def _histogram(engine, sigma, r0, v0):
    return adjoint.trajectory_histogram(r0, sigma, torch.ones(1, 1), engine, np.ones((1, 1), np.float32), v0)


def test_autograd_function_differentiates_its_own_pass():
    engine = OneTrajectory()
    s = [torch.full((1, 1), x, requires_grad=True) for x in (2.0, 3.0)]
    r0 = [torch.full((1, 3), x, requires_grad=True) for x in (1.0, 5.0)]
    v0 = np.ones((1, 3), np.float32)
    a, b = (_histogram(engine, s[k], r0[k], v0) for k in range(2))
    with torch.no_grad():
        r0[0] += 10.0           # a step of an optimizer: not what the pass was computed from
    with pytest.raises(gp._native.NativeError):
        _histogram(engine, torch.full((1, 1), -1.0), r0[0], v0)
    (a + 10 * b).sum().backward()
    assert s[0].grad.item() == 4.0 and s[1].grad.item() == 60.0
    assert r0[0].grad[0, 0].item() == 1.0 and r0[1].grad[0, 0].item() == 50.0


def _model(seed):
    conf = gp.Configuration(D=3)
    conf.make_lattice(gp.unit_cells.FCC, cells=[5, 5, 5], rho=1.2)
    conf['m'] = 1.0
    rng = np.random.default_rng(seed)
    conf.ptype[rng.permutation(conf.N)[:conf.N // 5]] = 1
    conf['r'] = conf['r'] + rng.uniform(-0.03, 0.03, conf['r'].shape).astype(np.float32)
    conf.randomize_velocities(temperature=0.8, seed=seed)
    return conf, adjoint.DifferentiableNVE(conf, dt=0.004, nsteps=20, cut=2.5 * np.array(KA_SIG), ckpt_every=10,
                                           rdf_every=5, bins=60, rmax=2.4, width=0.03)


@pytest.mark.gpu
def test_two_passes_then_both_gradients():
    conf, m = _model(3)
    r0 = torch.tensor(conf['r'])
    eps = torch.tensor(KA_EPS)

    def loss(s):
        return (m.rdf(r0, s, eps) ** 2).mean()

    start = [torch.tensor(KA_SIG) * f for f in (1.0, 0.97)]
    alone = []
    for x in start:
        s = x.clone().requires_grad_()
        loss(s).backward()
        alone.append(s.grad.numpy())
    s = [x.clone().requires_grad_() for x in start]
    first, second = loss(s[0]), loss(s[1])
    (first + second).backward()
    for got, ref in zip(s, alone):
        np.testing.assert_array_equal(got.grad.numpy(), ref)


@pytest.mark.gpu
def test_a_failed_pass_leaves_nothing_to_differentiate():
    conf, m = _model(4)
    params = np.stack([KA_SIG, KA_EPS, 2.5 * np.array(KA_SIG)], -1).astype(np.float32)
    m.engine.forward(params, conf['r'], conf['v'])
    bad = params.copy()
    bad[1, 1, 0] = -1.0     # refused after the constants of the other types have been replaced
    with pytest.raises(gp._native.NativeError, match="sigma"):
        m.engine.forward(bad, conf['r'], conf['v'])
    with pytest.raises(gp._native.NativeError, match="no forward pass"):
        m.engine.backward(np.ones((m.engine.ncls, m.bins)))
