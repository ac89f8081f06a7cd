"""Scalar rows whose columns are not all the device's: two quantities in one
column, columns of the caller's own, columns named outside the row.  What the
device does not hold stays as the caller has it, on every size's way through
the packed transfers."""
import numpy as np
import pytest

from gamdpy_amd import _native

pytestmark = pytest.mark.gpu

#                 u   w  lap  k  fsq  m   columns the device holds
CASES = [(3, (0, 0, -1, -1, -1, 1), [0, 1]),      # two quantities in column 0: as many names as columns
         (2, (0, 5, -1, -1, -1, 1), [0, 1]),      # column 5 of 2
         (4, (3, 1, -1, -1, -1, 0), [0, 1, 3]),
         (1, (-1, -1, -1, -1, -1, 0), [0])]


@pytest.mark.parametrize("N", [64, 1500, 70001])
@pytest.mark.parametrize("ns,sids,held", CASES)
def test_other_columns_stay(N, ns, sids, held):
    fields = {"N": N, "D": 3, "ntypes": 1, "box": [60.0] * 3, "pair_base": 0, "cutoff": 1, "max_cut": 2.5,
              "nblist_kind": 0, "skin": 0.3, "max_nbs": 32, "integrator": 0, "dt": 0.0, "compute_u": 1,
              "compute_w": 1, "pb": 64, "tp": 4, "nscalars": ns}
    fields.update(zip(("sid_u", "sid_w", "sid_lap", "sid_k", "sid_fsq", "sid_m"), sids))
    ctx = _native.Context(fields, np.array([[[1.0, 1.0, 2.5]]]))
    rng = np.random.default_rng(N)
    up = rng.normal(0.0, 1.0, (N, ns)).astype(np.float32)
    v = rng.normal(0.0, 1.0, (N, 3)).astype(np.float32)
    ctx.upload(r=np.zeros((N, 3)), v=v, f=v, scalars=up, ptype=np.zeros(N), r_im=np.zeros((N, 3)))
    out = np.full((N, ns), 7.0, np.float32)
    got_v = np.zeros_like(v)
    _native.check(ctx.lib.gmd_download(ctx.h, None, _native.fptr(got_v), None, _native.fptr(out), None, None))
    np.testing.assert_array_equal(got_v, v)
    for col in range(ns):
        np.testing.assert_array_equal(out[:, col], up[:, col] if col in held else 7.0, err_msg=str(col))
    sc = ctx.download()[3]
    for col in range(ns):
        np.testing.assert_array_equal(sc[:, col], up[:, col] if col in held else 0.0, err_msg=str(col))
