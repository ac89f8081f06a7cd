"""N-squared rebuilds that take one particle a wavefront (plans of one or two
rounds) and four (more): a particle's sums have one order for a size of block
(its tiles), so the forces and scalars have the same bits for every plan of
that size, and the neighbour sets are the oracle's.  With and without half lists, exclusions and bonds, and with
positions outside the box."""
import numpy as np
import pytest

import gamdpy_amd as gp
from helpers import KA_EPS, KA_SIG, plan, rows_from_array
from oracle import md_oracle as orc
from test_gpu_nsq_edges import _system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [256, 64])
@pytest.mark.parametrize("form", ["plain", "niii", "bonds", "outside"])
@pytest.mark.parametrize("N", [37, 256, 321, 1025])
def test_one_and_four_particles_a_wavefront(N, form, block):
    conf = _system(N, 1.0, N, form == "outside")
    func = gp.apply_shifted_potential_cutoff(gp.LJ_12_6_sigma_epsilon)
    excl, bonds = None, []
    if form == "bonds":
        b = gp.Bonds(gp.harmonic_bond_function, [[1.0, 100.0]], [[a, a + 1, 0] for a in range(0, N - 1, 2)])
        excl, bonds = b.get_exclusions(conf, max_number_exclusions=4), [b]
    pp = gp.PairPotential(func, params=[KA_SIG, KA_EPS, np.array(KA_SIG) * 1.5], max_num_nbs=200, exclusions=excl)
    rows = orc.nblist_nsquared(conf['r'], conf.simbox.lengths, float(pp.param_table()[1]), 0.5)
    if form == "bonds":
        rows = [np.setdiff1d(row, [i ^ 1]) if i ^ 1 < N else row for i, row in enumerate(rows)]
    first = None
    for tp in (64, 32, 16, 1):
        p = plan(tp=tp, pb=block // tp)
        p['UtilizeNIII'] = form == "niii"
        ev = gp.Evaluator(conf, [pp] + bonds, compute_plan=p)
        ev.evaluate()
        got = [conf[name].copy() for name in ('f', 'U', 'W')]
        if form != "niii":
            for x, y in zip(rows_from_array(ev.ctx.nblist()), rows):
                np.testing.assert_array_equal(x, y)
        first = first or got
        for x, y, name in zip(got, first, ('f', 'U', 'W')):
            np.testing.assert_array_equal(x, y, err_msg=f"{name}, tp {tp}")
