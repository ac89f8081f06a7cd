"""Pair counts of positions that are sorted first and of positions whose
numbering is in order already (lattice order; a context renumbered in cell
order), on both sides of the sizes where that makes a difference: the oracle's."""
import numpy as np
import pytest

import gamdpy_amd as gp
from gamdpy_amd import _native
from helpers import lj_pair_potential, plan
from oracle import c_oracle

pytestmark = pytest.mark.gpu


def _lattice(N, seed):
    rng = np.random.default_rng(seed)
    n = int(np.ceil((N / 4) ** (1 / 3)))
    r, box = gp.make_lattice(gp.unit_cells.FCC, [n, n, n], rho=0.8)
    r = r[np.sort(rng.permutation(len(r))[:N])] + rng.uniform(-0.1, 0.1, (N, 3))
    return r.astype(np.float32), np.float32(box), rng


@pytest.mark.parametrize("N", [8191, 8192, 8211, 32769, 65537])
def test_host_positions(N):
    r, box, rng = _lattice(N, N)
    pt = rng.integers(0, 2, N).astype(np.int32)
    ref = c_oracle.rdf_counts(r, pt, box, 200, 2)
    rdf = _native.RdfHandle(N, 2, 200)
    for p in (np.arange(N), rng.permutation(N), np.arange(N)):
        assert np.array_equal(rdf.compute_host(r[p], pt[p], box).astype(np.int64), ref)
        if N <= 65536:
            assert np.array_equal(_native.rdf_counts_noalloc(r[p], pt[p], box, 2, 200).astype(np.int64), ref)


def test_renumbered_context():
    N = 8209
    r, box, rng = _lattice(N, 7)
    conf = gp.Configuration(D=3)
    conf['r'] = r[rng.permutation(N)]
    conf.simbox = gp.Orthorhombic(3, box)
    conf['m'] = 1.0
    sim = gp.Simulation(conf, lj_pair_potential(), gp.NVE(dt=0.001), [], num_timeblocks=1, steps_per_timeblock=2,
                        compute_plan=plan(tp=4, nblist='linked lists'), storage='memory', steps_in_kernel_test=0)
    calc = gp.CalculatorRadialDistribution(conf, bins=200)
    conf.copy_to_device()
    for steps in (0, 2):      # in the caller's numbering, in cell order
        sim.ctx.run(0.0, steps)
        assert sim.ctx.reorder_stats()[0] == (steps > 0)
        calc.update()
        ref = c_oracle.rdf_counts(sim.ctx.download()[0], conf.ptype, box, 200, 1)
        assert np.array_equal(calc.rdf_list[-1].astype(np.int64), ref)
