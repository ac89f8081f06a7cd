"""Pair counts at the sizes where the histogram kernel changes form: around the
16 particles of a group and the 64 of a chunk, the odd middle row of chunks,
the sizes from which particles are sorted into cells, distances exactly on a
bin's edge, anisotropic boxes, everything in one place.  Counts are whole
numbers and equal the oracle's."""
import numpy as np
import pytest

from gamdpy_amd import _native
from oracle import c_oracle

pytestmark = pytest.mark.gpu


def _positions(kind, N, box, rng):
    box = np.asarray(box, np.float32)
    if kind == "uniform":
        return (rng.uniform(-0.5, 0.5, (N, 3)) * box).astype(np.float32)
    if kind == "grid":   # distances on the bins' edges, many of them equal, and particles at +-L/2
        return (rng.integers(-8, 9, (N, 3)) / 16.0 * box).astype(np.float32)
    if kind == "cluster":   # all in a corner's cell, across the periodic boundary
        r = (0.49 + rng.uniform(0.0, 0.02, (N, 3))) * box
        return (r - box * (r > 0.5 * box)).astype(np.float32)
    raise ValueError(kind)


@pytest.mark.parametrize("kind", ["uniform", "grid", "cluster"])
@pytest.mark.parametrize("N,nt,bins,box", [
    (1, 1, 5, (4.0, 4.0, 4.0)), (2, 2, 64, (16.0, 16.0, 16.0)), (16, 1, 64, (16.0, 16.0, 16.0)),
    (17, 2, 100, (9.0, 7.0, 11.0)), (63, 1, 64, (16.0, 16.0, 16.0)), (65, 3, 33, (16.0, 16.0, 16.0)),
    (129, 2, 1000, (5.0, 5.0, 5.0)), (1000, 2, 64, (16.0, 32.0, 16.0)), (8191, 1, 3000, (16.0, 16.0, 16.0)),
    (8192, 2, 1000, (16.0, 16.0, 16.0)), (8209, 3, 64, (16.0, 16.0, 16.0)), (33001, 2, 500, (30.0, 40.0, 24.0))])
def test_rdf_counts_at_edges(N, nt, bins, box, kind):
    rng = np.random.default_rng(N + bins)
    r = _positions(kind, N, box, rng)
    pt = rng.integers(0, nt, N).astype(np.int32)
    ref = c_oracle.rdf_counts(r, pt, np.array(box, np.float32), bins, nt)
    rdf = _native.RdfHandle(N, nt, bins)
    print(kind, N, nt, bins, ref.sum(), flush=True)
    for _ in range(2):
        assert np.array_equal(rdf.compute_host(r, pt, box).astype(np.int64), ref)
    if nt * nt * bins <= 4096:
        assert np.array_equal(_native.rdf_counts_noalloc(r, pt, box, nt, bins).astype(np.int64), ref)
