"""Host arrays to and from the device: small systems (the packing kernels read
and write pinned memory), larger ones (through a device buffer) and ones whose
packed arrays pass through the pinned buffer in halves, in the caller's
numbering also where the particles are renumbered.  What is uploaded comes
back bit for bit, and a partial upload leaves everything else as it was."""
import numpy as np
import pytest

import gamdpy_amd as gp
from helpers import plan

pytestmark = pytest.mark.gpu


def _conf(N, seed=0):
    rng = np.random.default_rng(seed)
    n = int(np.ceil((N / 4) ** (1 / 3)))
    r, box = gp.make_lattice(gp.unit_cells.FCC, [n, n, n], rho=0.8)
    conf = gp.Configuration(D=3)
    conf['r'] = (r[rng.permutation(len(r))[:N]] + 0.1).astype(np.float32)
    conf.simbox = gp.Orthorhombic(3, box)
    conf['m'] = rng.uniform(1.0, 2.0, N).astype(np.float32)
    conf['v'] = rng.normal(0.0, 1.0, (N, 3)).astype(np.float32)
    conf['f'] = rng.normal(0.0, 1.0, (N, 3)).astype(np.float32)
    conf.ptype = rng.integers(0, 2, N).astype(np.int32)
    conf.r_im = rng.integers(-5, 5, (N, 3)).astype(np.int32)
    return conf


def _pair():
    return gp.PairPotential(gp.apply_shifted_potential_cutoff(gp.LJ_12_6_sigma_epsilon),
                            params=[np.ones((2, 2)), np.ones((2, 2)), 2.0 * np.ones((2, 2))], max_num_nbs=256)


@pytest.mark.parametrize("N,nblist", [(500, 'N squared'), (1024, 'N squared'), (1025, 'N squared'),
                                      (5000, 'linked lists'), (100003, 'linked lists')])
def test_round_trip_and_partial_uploads(N, nblist):
    conf = _conf(N)
    sim = gp.Simulation(conf, _pair(), gp.NVE(dt=0.0), [], num_timeblocks=1, steps_per_timeblock=2,
                        compute_plan=plan(tp=4, nblist=nblist), storage='memory', steps_in_kernel_test=0)
    ctx = sim.ctx
    rng = np.random.default_rng(1)
    sc = rng.normal(0.0, 1.0, conf.scalars.shape).astype(np.float32)
    sc[:, conf.sid['m']] = conf['m']
    want = dict(r=conf['r'].copy(), v=conf['v'].copy(), f=conf['f'].copy(), scalars=sc, ptype=conf.ptype.copy(),
                r_im=conf.r_im.copy())
    names = ('r', 'v', 'f', 'scalars', 'ptype', 'r_im')

    def check():
        for name, got in zip(names, ctx.download()):
            np.testing.assert_array_equal(got, want[name], err_msg=name)

    ctx.upload(**want)
    check()
    # time steps of length zero: nothing moves, but with linked lists the
    # particles are renumbered
    ctx.run(0.0, 2)
    assert ctx.reorder_stats()[0] == (nblist == 'linked lists')
    r, v, _, _, pt, im = ctx.download()
    for got, name in ((r, 'r'), (v, 'v'), (pt, 'ptype'), (im, 'r_im')):
        np.testing.assert_array_equal(got, want[name], err_msg=name)
    ctx.upload(**want)
    for name, new in (('r', want['r'][::-1]), ('ptype', 1 - want['ptype']), ('v', -want['v']), ('f', 2 * want['f']),
                      ('r_im', want['r_im'] + 1), ('scalars', np.float32(1.5) * sc)):
        want[name] = np.ascontiguousarray(new)
        ctx.upload(**{name: want[name]})
        check()
    # into the caller's own arrays
    rows = [np.zeros((N, 3), np.float32) for _ in range(3)]
    ctx.download(rows)
    for got, name in zip(rows, ('r', 'v', 'f')):
        np.testing.assert_array_equal(got, want[name])


def test_batch_fetch_equals_single_downloads():
    confs = [_conf(N, seed=N) for N in (600, 1500, 7000)]
    for c in confs:
        c['m'] = 1.0
        c['v'] = 0.1 * c['v']
    batch = gp.BatchedSimulation([gp.Replica(c, _pair(), gp.NVE(dt=0.002)) for c in confs], 1, 30, tp=2,
                                 driver='graph')
    batch.integrate_self(0.0, 30)
    plain = [ctx.download() for ctx in batch.batch.contexts]
    batch.batch.fetch()
    for ctx, ref in zip(batch.batch.contexts, plain):
        for got, x in zip(ctx.download(), ref):
            np.testing.assert_array_equal(got, x)
