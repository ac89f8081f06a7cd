"""What the differentiable trajectory refuses and what it falls back to."""
import numpy as np
import pytest
import torch

from gamdpy_amd import _native
from gamdpy_amd.adjoint import AdjointEngine

pytestmark = pytest.mark.gpu


def _engine(N, L, nsteps=1, **kw):
    kw = dict(dict(ckpt_every=5, rdf_every=5, bins=20, rmax=3.0, width=0.02), **kw)
    return AdjointEngine(N, 1, [L] * 3, 0.0, nsteps, np.zeros(N, np.int32), np.ones(N, np.float32), **kw)


LJ = np.array([[[1.0, 1.0, 1.7]]], np.float32)


def test_frame_lists_too_long_for_the_gradient_are_refused_by_the_forward_pass():
    """A droplet: 146 neighbours a particle, room for twice the mean of a
    homogeneous system and 64 more (here 96).  Half of them would fit."""
    n, L = 7, 40.0
    r = np.stack(np.meshgrid(*[np.arange(n) * 0.95 - 0.95 * (n - 1) / 2] * 3, indexing="ij"), -1).reshape(-1, 3)
    d = np.linalg.norm(r[:, None] - r[None], axis=-1)
    longest = int((d < 3.0 + 5 * 0.02).sum(1).max()) - 1
    assert 96 < longest < 192 and int((d < 2.2).sum(1).max()) - 1 <= 64   # (the step's own lists fit)
    eng = _engine(len(r), L)
    with pytest.raises(_native.NativeError, match=f"frame list of {longest} entries"):
        eng.forward(LJ, r, np.zeros_like(r))


def test_a_trajectory_that_leaves_no_room_for_the_rest_is_not_kept():
    """Device memory for everything but 50 MB of: a trajectory of 963 MB, lists
    of 77 MB, histograms of 75 MB and 23 MB of vectors.  The checkpoints (170 MB)
    fit."""
    room = (963 + 175 - 50) << 20
    held = []
    for share in (0.9, 1.0, 1.0):
        extra = int(share * (torch.cuda.mem_get_info()[0] - room)) >> 21 << 21
        if extra > 0:
            held.append(torch.empty(extra, dtype=torch.uint8, device="cuda"))
    free = torch.cuda.mem_get_info()[0]
    if not abs(free - room) < (20 << 20):
        pytest.skip(f"{free >> 20} MB of device memory free instead of {room >> 20}")
    try:
        eng = _engine(200_000, 55.0, nsteps=300, ckpt_every=20, rmax=1.0, bins=3000)
        eng.close()
    finally:
        del held
        torch.cuda.empty_cache()


def test_checkpoints_by_choice():
    """keep_trajectory=False: the checkpoints' memory, the same bits."""
    n, nsteps = 27, 2000
    L = n * 1.1
    rng = np.random.default_rng(2)
    r = np.stack(np.meshgrid(*[np.arange(n) * 1.1 - L / 2 + 0.5] * 3, indexing="ij"), -1).reshape(-1, 3)
    r = (r + rng.uniform(-0.05, 0.05, r.shape)).astype(np.float32)
    v = rng.normal(0.0, 0.5, r.shape).astype(np.float32)
    used = []
    for keep in (True, False):
        before = torch.cuda.mem_get_info()[0]
        eng = _engine(n ** 3, L, nsteps=nsteps, ckpt_every=50, keep_trajectory=keep)
        used.append(before - torch.cuda.mem_get_info()[0])
        eng.close()
    assert used[0] - used[1] > 16 * (nsteps - 200) * n ** 3   # (checkpoints: 131 steps' worth)
    got = []
    for keep in (True, False):
        eng = AdjointEngine(n ** 3, 1, [L] * 3, 0.004, 12, np.zeros(n ** 3, np.int32), np.ones(n ** 3, np.float32),
                            ckpt_every=5, rdf_every=4, bins=20, rmax=2.0, width=0.05, keep_trajectory=keep)
        H = eng.forward(LJ, r, v)
        got.append((H,) + eng.backward(H))
        eng.close()
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)


def test_checkpoints_without_room_leave_the_handle_as_it_was():
    """A segment of 10^8 steps has no room: an error, and the trajectory is kept
    on; a handle that never had room for either refuses to be made."""
    rng = np.random.default_rng(3)
    r = np.stack(np.meshgrid(*[np.arange(12) * 1.1 - 6.6] * 3, indexing="ij"), -1).reshape(-1, 3)
    r = (r + rng.uniform(-0.05, 0.05, r.shape)).astype(np.float32)
    N, far = len(r), 10 ** 8
    eng = _engine(N, 13.2, nsteps=10, ckpt_every=far)
    ref = _engine(N, 13.2, nsteps=10, ckpt_every=100)
    want = ref.forward(LJ, r, 0 * r)
    np.testing.assert_array_equal(eng.forward(LJ, r, 0 * r), want)
    with pytest.raises(_native.NativeError, match="memory"):
        _native.check(eng.lib.gmd_adj_use_checkpoints(eng.h), "gmd_adj_use_checkpoints")
    with pytest.raises(_native.NativeError, match="no forward pass"):   # dropped, as the call says
        eng.backward(want)
    np.testing.assert_array_equal(eng.forward(LJ, r, 0 * r), want)
    for a, b in zip(eng.backward(want), ref.backward(want)):
        np.testing.assert_array_equal(a, b)
    with pytest.raises(_native.NativeError, match="memory"):
        _engine(N, 13.2, nsteps=10, ckpt_every=far, keep_trajectory=False)
