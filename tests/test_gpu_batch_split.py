"""Which batches split their rebuild steps, told by the blocks of a launch (a
split replica brings the blocks of its rebuild steps, an unsplit one those of
its list steps; the grid is a multiple of 8): the comparisons of split steps
with unsplit ones elsewhere compare what they say."""
import numpy as np
import pytest

import gamdpy_amd as gp
from test_gpu_rebuild_grid import CELLS, _batch

pytestmark = pytest.mark.gpu

NVT = lambda: gp.NVT(temperature=2.0, tau=0.2, dt=0.004)  # noqa: E731
NVE = lambda: gp.NVE(dt=0.004)  # noqa: E731


@pytest.mark.parametrize("integ", [NVT, NVE], ids=["NVT", "NVE"])
@pytest.mark.parametrize("driver,tp,cells,split", [
    ("graph", 1, CELLS, True), ("graph", 32, [[12, 12, 12]] * 4, False), ("persistent", 1, CELLS, False)])
def test_grid_tells_the_split(driver, tp, cells, split, integ):
    batch, reps = _batch(driver, tp, integ, 2, lambda: [], cells)
    n, grid = batch.batch.size()
    assert n == len(cells)
    blocks = sum(-(-r.configuration.N * tp // 256) for r in reps) if batch.blocks is None else int(np.sum(batch.blocks))
    if split:
        assert grid > blocks + 7
    else:
        assert blocks <= grid <= blocks + 7
