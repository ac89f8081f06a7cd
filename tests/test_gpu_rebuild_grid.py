"""Batches whose rebuild steps are split over more blocks than their list steps:
thermostat, barostat, momentum reset and saver rows agree with the persistent
driver (one grid for every step) to float32 rounding: 1e-7 of sums and
positions, grown by less than ten in 45 steps and added less than 45 times.
The kinetic sum of a split step has the bits of an unsplit one.  Lists and
forces of a split step against the oracle."""
import numpy as np
import pytest

import gamdpy_amd as gp
from helpers import ka_fcc, ka_pair_potential, rows_from_array
from oracle import md_oracle as orc

pytestmark = pytest.mark.gpu

# just past the smallest linked-list grid, linked lists, N squared of one block and a few
CELLS = [[8, 7, 7], [12, 12, 12], [5, 5, 5], [4, 4, 4]]


def _batch(driver, tp, integ, steps, actions, cells=CELLS):
    reps = [gp.Replica(ka_fcc(c, T=2.0, seed=k, jitter=0.05), ka_pair_potential(), integ(), actions())
            for k, c in enumerate(cells)]
    batch = gp.BatchedSimulation(reps, num_timeblocks=1, steps_per_timeblock=steps, tp=tp, skin=0.25, driver=driver)
    for _ in batch.run_timeblocks():
        pass
    return batch, reps


@pytest.mark.parametrize("tp,cells", [(1, CELLS),
                                      (32, CELLS),                 # more list blocks than cells or particles need
                                      (32, [[12, 12, 12]] * 4)])   # enough list blocks that no rebuild is split
@pytest.mark.parametrize("integ", [lambda: gp.NVT(temperature=2.0, tau=0.2, dt=0.004),
                                   lambda: gp.NPT_Atomic(temperature=2.0, tau=0.4, pressure=20.0, tau_p=20, dt=0.002)],
                         ids=["NVT", "NPT"])
def test_two_grids(tp, cells, integ):
    actions = lambda: [gp.ScalarSaver(3), gp.MomentumReset(7)]  # noqa: E731
    a, ra = _batch('graph', tp, integ, 45, actions, cells)
    b, rb = _batch('persistent', tp, integ, 45, actions, cells)
    for x, y, oa, ob in zip(ra, rb, a.outputs, b.outputs):
        assert x.ctx.nbflag()[2] == y.ctx.nbflag()[2] >= 3
        ca, cb = x.configuration, y.configuration
        L = ca.simbox.lengths
        np.testing.assert_allclose(L, cb.simbox.lengths, rtol=1e-5)
        d = ca['r'] - cb['r']
        assert np.max(np.abs(d - L * np.round(d / L))) < 1e-4
        np.testing.assert_allclose(oa["scalars"][0], ob["scalars"][0], rtol=1e-4, atol=1e-4 * ca.N)


def test_rebuild_alone():
    """The list built at step 0 (tp = 1), and the forces of a run of no steps."""
    _, reps = _batch('graph', 1, lambda: gp.NVE(dt=0.004), 0, lambda: [])
    for r in reps:
        conf = r.configuration
        table, max_cut = r.interaction.param_table()
        rows = orc.nblist_nsquared(conf['r'], conf.simbox.lengths, float(max_cut), 0.25)
        for x, y in zip(rows_from_array(r.ctx.nblist()), rows):
            np.testing.assert_array_equal(x, y)
        f, U, W, _ = orc.pair_forces(conf['r'], conf.ptype, conf.simbox.lengths, table, rows)
        for got, ref in ((conf['f'], f), (conf['U'], U), (conf['W'], W)):
            assert np.max(np.abs(got - ref)) < 1e-5 * np.max(np.abs(ref))


def test_split_keeps_the_bits():
    """With a saver row every step no rebuild is split, without one all are:
    the same trajectory, bit for bit (NVT, tp = 1: blocks of several rounds)."""
    nvt = lambda: gp.NVT(temperature=2.0, tau=0.2, dt=0.004)  # noqa: E731
    _, ra = _batch('graph', 1, nvt, 45, lambda: [])
    _, rb = _batch('graph', 1, nvt, 45, lambda: [gp.ScalarSaver(1)])
    for x, y in zip(ra, rb):
        assert x.ctx.nbflag()[2] == y.ctx.nbflag()[2] >= 3
        assert np.array_equal(x.integrator.thermostat_state, y.integrator.thermostat_state)
        for name in ('r', 'v', 'f'):
            assert np.array_equal(x.configuration[name], y.configuration[name]), name
