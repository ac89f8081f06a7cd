"""The list builds' forms: with the boxes of chunks (a numbering in lattice
order in a box several list radii long), without them (the same particles in no
order), inside the step kernels and in launches of their own (from 8000
particles).  Histograms against the float64 C program, and both numberings'
gradients against each other; tolerances as between float32 and float64
trajectories (1e-3 and 1e-2)."""
import numpy as np
import pytest
import torch

import gamdpy_amd as gp
from gamdpy_amd.adjoint import DifferentiableNVE
from helpers import KA_EPS, KA_SIG
from oracle import c_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,N", [([4, 4, 17], 1025), ([4, 4, 20], 1279), ([13, 13, 12], 7999), ([13, 13, 12], 8003)])
def test_numberings_agree(cells, N):
    rng = np.random.default_rng(N)
    r, box = gp.make_lattice(gp.unit_cells.FCC, cells, rho=1.0 * 4 * np.prod(cells) / N)
    order = np.lexsort((r[:, 0], r[:, 1], r[:, 2]))       # slabs along z: compact chunks in a long box
    r = r[order][np.sort(rng.permutation(len(r))[:N])] + rng.uniform(-0.03, 0.03, (N, 3))
    r = r.astype(np.float32)
    pt = np.zeros(N, np.int32)
    pt[rng.permutation(N)[:N // 5]] = 1
    v = rng.normal(0.0, 1.7, (N, 3)).astype(np.float32)
    v -= v.mean(0)
    sig, eps = np.array(KA_SIG), np.array(KA_EPS)
    traj = dict(dt=0.004, nsteps=40, rdf_every=20, bins=50, rmax=2.0, width=0.03)
    Hc, _ = c_oracle.adj_histogram_f64(r.astype(np.float64), v.astype(np.float64), np.ones(N), pt,
                                       np.float32(box), np.stack([sig, eps, 2.3 * sig], -1), traj['dt'],
                                       traj['nsteps'], traj['rdf_every'], traj['bins'], traj['rmax'], traj['width'])
    got = []
    for p in (np.arange(N), rng.permutation(N)):
        conf = gp.Configuration(D=3)
        conf['r'] = r[p]
        conf.simbox = gp.Orthorhombic(3, np.float32(box))
        conf['m'] = 1.0
        conf['v'] = v[p]
        conf.ptype = pt[p]
        m = DifferentiableNVE(conf, cut=2.3 * sig, ckpt_every=100, **traj)
        r0 = torch.tensor(conf['r'], requires_grad=True)
        s, e = (torch.tensor(x, requires_grad=True) for x in (sig, eps))
        H = m.histogram(r0, s, e)
        ((H / H.detach().max()) ** 2).sum().backward()
        print(N, np.abs(H.detach().numpy() - Hc).max() / Hc.max())
        assert np.abs(H.detach().numpy() - Hc).max() <= 1e-3 * Hc.max()
        back = np.empty_like(r)
        back[p] = r0.grad.numpy()
        got.append((back, s.grad.numpy(), e.grad.numpy()))
    for a, b in zip(*got):
        print(np.linalg.norm(a - b) / np.linalg.norm(b))
        assert np.linalg.norm(a - b) <= 1e-2 * np.linalg.norm(b)
