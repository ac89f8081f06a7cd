"""Pair counts where some positions are not numbers or infinite (a simulation
that has blown up): such particles have no pairs, and everyone else's pairs are
counted as they are without them.  One of them stands first in a group of 16
and in a chunk of 64, whose boxes are laid out around their first particle."""
import numpy as np
import pytest

from gamdpy_amd import _native
from oracle import c_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("N,at", [(40, [16]), (129, [64, 128]), (1000, [0, 80, 999]), (9000, [0, 64, 4000])])
def test_others_pairs_are_counted(N, at, bad):
    rng = np.random.default_rng(N)
    box = np.array([12.0, 10.0, 14.0], np.float32)
    r = (rng.uniform(-0.5, 0.5, (N, 3)) * box).astype(np.float32)
    r[at, 0] = bad
    pt = rng.integers(0, 2, N).astype(np.int32)
    good = np.setdiff1d(np.arange(N), at)
    ref = c_oracle.rdf_counts(r[good], pt[good], box, 100, 2)
    rdf = _native.RdfHandle(N, 2, 100)
    assert np.array_equal(rdf.compute_host(r, pt, box).astype(np.int64), ref)
    assert np.array_equal(_native.rdf_counts_noalloc(r, pt, box, 2, 100).astype(np.int64), ref)
