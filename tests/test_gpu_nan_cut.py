"""A type pair whose cut is not a number has no interactions, in the step that
builds the list as in the steps that use it."""
import numpy as np
import pytest

from gamdpy_amd import _native
from helpers import KA_EPS, KA_SIG, ka_fcc
from oracle import md_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,kind,tp", [([5, 5, 5], 0, 4), ([5, 5, 5], 0, 64), ([8, 7, 7], 1, 4)])
def test_no_pairs(cells, kind, tp):
    conf = ka_fcc(cells, seed=3, jitter=0.05)
    N = conf.N
    table = np.stack([KA_SIG, KA_EPS, 2.5 * np.array(KA_SIG)], -1).astype(np.float32)
    none = table.copy()
    table[1, 1, 2] = np.nan
    none[1, 1, 2] = 1e-3
    ctx = _native.Context({"N": N, "D": 3, "ntypes": 2, "box": conf.simbox.lengths, "pair_base": 0, "cutoff": 1,
                           "max_cut": 2.5, "nblist_kind": kind, "skin": 0.3, "max_nbs": 300, "integrator": 0,
                           "dt": 0.0, "compute_u": 1, "compute_w": 1, "pb": 256 // tp, "tp": tp, "nscalars": 1,
                           "sid_u": 0, "sid_w": -1, "sid_lap": -1, "sid_k": -1, "sid_fsq": -1, "sid_m": -1}, table)
    ctx.upload(r=conf['r'], v=conf['v'], ptype=conf.ptype, scalars=np.zeros((N, 1)), f=conf['f'], r_im=conf.r_im)
    rows = orc.nblist_nsquared(conf['r'], conf.simbox.lengths, 2.5, 0.3)
    f_ref, u_ref = orc.pair_forces(conf['r'], conf.ptype, conf.simbox.lengths, none, rows)[:2]
    for rebuild in (True, False):
        if rebuild:
            ctx.force_rebuild()
        ctx.evaluate()
        _, _, f, sc, _, _ = ctx.download()
        assert np.max(np.abs(f - f_ref)) < 1e-5 * np.max(np.abs(f_ref))
        assert np.max(np.abs(sc[:, 0] - u_ref)) < 1e-5 * np.max(np.abs(u_ref))
