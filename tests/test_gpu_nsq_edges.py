"""N-squared rebuild at the edges of its tiling: a wavefront takes four
particles at a time and a block tiles of blockDim.x positions, so sizes just
below and above a tile, one particle per wavefront and many, blocks of one
wavefront, a box too small for the short minimum image, and positions outside
the box.  Neighbour sets equal to the oracle's; forces, U and W within the
parity tests' 1e-5 of the largest value."""
import numpy as np
import pytest

import gamdpy_amd as gp
from oracle import md_oracle as orc
from helpers import KA_EPS, KA_SIG, plan, rows_from_array

pytestmark = pytest.mark.gpu


def _system(N, rho, seed, outside):
    rng = np.random.default_rng(seed)
    n = int(np.ceil((N / 4) ** (1 / 3)))
    r, box = gp.make_lattice(gp.unit_cells.FCC, [n, n, n], rho=rho * 4 * n ** 3 / N)
    r = r[np.sort(rng.permutation(len(r))[:N])] + rng.uniform(-0.05, 0.05, (N, 3)) + 0.1
    box = np.float32(box)
    r -= box * np.round(r / box)
    if outside:
        r[::7] += box * np.array([1.0, 0.0, 0.0])
    conf = gp.Configuration(D=3)
    conf['r'] = r.astype(np.float32)
    conf.simbox = gp.Orthorhombic(3, box)
    conf['m'] = 1.0
    conf.ptype[rng.permutation(N)[:N // 5]] = 1
    return conf


@pytest.mark.parametrize("N,tp,pb,rho,outside", [
    (37, 16, 16, 0.1, False),     # less than a wavefront of particles
    (256, 16, 16, 1.0, False),    # exactly one tile
    (257, 2, 128, 1.0, False),    # one position in the last tile; 32 rounds
    (321, 64, 4, 1.0, False),     # one particle a wavefront
    (500, 16, 4, 1.0, False),     # blocks of one wavefront: tiles of 64
    (300, 1, 192, 1.0, False),    # blocks of three wavefronts, 64 rounds
    (108, 16, 16, 1.0, False),    # list radius above half the box
    (1025, 8, 32, 1.0, True),     # positions outside the box
])
def test_nsq_rebuild_edges(N, tp, pb, rho, outside):
    conf = _system(N, rho, N, outside)
    func = gp.apply_shifted_potential_cutoff(gp.LJ_12_6_sigma_epsilon)
    cut = np.array(KA_SIG) * 2.0
    pp = gp.PairPotential(func, params=[KA_SIG, KA_EPS, cut], max_num_nbs=400)
    ev = gp.Evaluator(conf, pp, compute_plan=plan(tp=tp, pb=pb))
    ev.evaluate()
    table, max_cut = pp.param_table()
    rows = orc.nblist_nsquared(conf['r'], conf.simbox.lengths, float(max_cut), 0.5)
    got = rows_from_array(ev.ctx.nblist())
    for i, (a, b) in enumerate(zip(got, rows)):
        np.testing.assert_array_equal(a, b, err_msg=f"particle {i}")
    f, U, W, _ = orc.pair_forces(conf['r'], conf.ptype, conf.simbox.lengths, table, rows)
    for name, got_x, ref in (("f", conf['f'], f), ("U", conf['U'], U), ("W", conf['W'], W)):
        err = np.max(np.abs(got_x - ref)) / max(np.max(np.abs(ref)), 1e-30)
        print(f"N={N} tp={tp} {name}: {err:.2e}")
        assert err < 1e-5
