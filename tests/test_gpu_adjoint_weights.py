"""The frame histogram adds every kernel weight with all its bits: isolated
pairs whose distances leave weights of 1e-8 to 1 in the bins, against the same
float32 arithmetic on the host.  The largest difference allowed is that of the
exponential's last bits (2^-22 relative to e^(-x^2 / 2 w^2), before the floor
e^-12.5 is taken off), and the float32 rounding of the weight itself; a sum
held in 2^-32 is off by up to 2.3e-10 a pair, a thousand times more for a
weight at the floor."""
import numpy as np
import pytest

from gamdpy_amd.adjoint import AdjointEngine

pytestmark = pytest.mark.gpu
F = np.float32


def _weights(d, bins, rmax, width):
    """float32 as the kernel has it -> e (bins,), weight (bins,) of distance d"""
    dr, wid = F(rmax) / F(bins), F(width)
    inv_w2 = F(1.0) / (wid * wid)
    k = np.arange(bins, dtype=np.float32)
    x = F(np.float64(d) - (k + F(0.5)).astype(np.float64) * np.float64(dr))
    y = ((F(-0.5) * x) * x) * inv_w2
    e = np.exp2((y * F(1.4426950408889634)).astype(np.float64)).astype(np.float32)
    kv = e - F(np.exp(F(-12.5)))
    return np.where(kv > 0, e, F(0)), np.where(kv > 0, kv, F(0))


def test_small_weights_keep_their_bits():
    bins, rmax, width, L = 50, 2.0, 0.03, 60.0
    rng = np.random.default_rng(1)
    # five pairs in one bin's tail, and 15 anywhere
    d = np.concatenate([0.02 + 0.04 * 20 + 5 * 0.03 - np.array([1e-6, 1e-5, 1e-4, 1e-3, 3e-3]),
                        rng.uniform(0.5, 1.9, 15)])
    base = np.stack(np.meshgrid(*[np.arange(5) * 11.0 - 22.0] * 3, indexing="ij"), -1).reshape(-1, 3)[:len(d)]
    r = np.empty((2 * len(d), 3), np.float32)
    r[0::2] = base
    r[1::2] = base + np.stack([d, 0 * d, 0 * d], -1)
    N = len(r)
    eng = AdjointEngine(N, 1, [L] * 3, 0.0, 1, np.zeros(N, np.int32), np.ones(N, np.float32), ckpt_every=1,
                        rdf_every=2, bins=bins, rmax=rmax, width=width)
    H = eng.forward(np.array([[[1.0, 1.0, 2.5]]]), r, np.zeros((N, 3)))[0]
    ref, room = np.zeros(bins), np.zeros(bins)
    for a, b in zip(r[0::2], r[1::2]):
        e, kv = _weights(np.abs(a[0] - b[0]), bins, rmax, width)
        ref += kv.astype(np.float64)
        room += e.astype(np.float64) * 2.0 ** -22
    print(np.abs(H - ref).max(), (np.abs(H - ref) / np.maximum(room, 1e-300)).max(), ref[ref > 0].min())
    assert ref[ref > 0].min() < 1e-6
    assert np.all(np.abs(H - ref) <= room)
