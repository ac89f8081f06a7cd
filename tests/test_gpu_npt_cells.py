"""A barostat that scales the box by several cell lengths in one step (a bad
start): the cell lists of the next step are those of the new box, so its
neighbour lists and forces are the oracle's."""
import numpy as np
import pytest

import gamdpy_amd as gp
from helpers import lj_pair_potential, plan, rows_from_array
from oracle import md_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rate,growth", [(60.0, 1.1), (200.0, 1.3)])
def test_lists_after_a_step_that_scales_the_box(rate, growth):
    conf = gp.Configuration(D=3)
    conf.make_lattice(gp.unit_cells.FCC, cells=[9, 9, 9], rho=0.7)
    conf['m'] = 1.0
    rng = np.random.default_rng(5)
    conf['r'] = conf['r'] + rng.uniform(-0.1, 0.1, conf['r'].shape).astype(np.float32)
    conf.randomize_velocities(temperature=1.0, seed=5)
    box = conf.simbox.lengths.copy()
    pp = lj_pair_potential(max_nbs=300)
    itg = gp.NPT_Atomic(temperature=1.0, tau=0.4, pressure=2.0, tau_p=20.0, dt=0.002)
    sim = gp.Simulation(conf, pp, itg, [], num_timeblocks=1, steps_per_timeblock=1,
                        compute_plan=plan(tp=4, nblist='linked lists'), storage='memory', steps_in_kernel_test=0)
    itg.barostat_state[0] = rate
    before = sim.ctx.nbflag()[2]
    for _ in sim.run_timeblocks():
        pass
    L = conf.simbox.lengths
    assert np.all(np.abs(L / box / growth - 1) < 0.03)
    assert sim.ctx.nbflag()[2] == before + 2      # the scaling moves the outer particles past the skin
    table, max_cut = pp.param_table()
    rows = orc.nblist_nsquared(conf['r'], L, float(max_cut), 0.5)
    for x, y in zip(rows_from_array(sim.ctx.nblist()), rows):
        np.testing.assert_array_equal(x, y)
    f_ref = orc.pair_forces(conf['r'], conf.ptype, L, table, rows)[0]
    assert np.max(np.abs(conf['f'] - f_ref)) < 1e-5 * np.max(np.abs(f_ref))
