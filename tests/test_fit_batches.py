"""What a band fit asks of the solver, counted by a stand-in for it: the reference point of the energy zero rides on
the k-points' batch, and its valence states are not solved for at every k-point of a large set."""
import types

import numpy as np
import pytest

from picomax_amd import autograd


class _Solver:
    """Levels e_n(k) = a0 n + a1 |k|^2 with their gradient; counts levels and vectors."""

    def __init__(self):
        self.vg = np.array([[1.5, 0.25]])
        self.levels = self.vectors = 0

    def bands(self, K, nband, offset):
        self.levels += len(K) * nband
        return self.vg[0, 0] * np.arange(nband)[None, :] + self.vg[0, 1] * (K ** 2).sum(1)[:, None] - offset

    def ref_energy(self, k, n):
        e = self.bands(np.asarray(k)[None, :], n + 1, 0.0)[0]
        return (e[n - 1] + e[n]) / 2

    def grad_bands(self, K, nband, g):
        assert g.shape == (len(K), nband)
        self.vectors += len(K) * nband
        return np.array([[(g * np.arange(nband)).sum(), (g * (K ** 2).sum(1)[:, None]).sum()]])


@pytest.mark.parametrize("nk", [1, 7, 8, 9, 16, 17, 40])
@pytest.mark.parametrize("nband,nvalence", [(1, 18), (4, 8), (12, 8)])
def test_vectors_asked_for(nk, nband, nvalence):
    m = autograd.BandModel.__new__(autograd.BandModel)
    m.ctx, m.sys, m.natom, m.nv = _Solver(), types.SimpleNamespace(npw=50), 1, 2
    m.refpoint, m.nvalence, m.batch = np.array([0.1, 0.0, 0.2]), nvalence, 8
    r = np.random.default_rng(nk)
    K, g = r.uniform(-0.5, 0.5, (nk, 3)), r.normal(size=(nk, nband))
    h = 1e-3  # the stand-in is linear in its parameters: differences are exact
    got, want = m.grad(K, nband, g), np.zeros((1, 2))
    vectors = m.ctx.vectors
    for i in range(2):
        d = []
        for sgn in (1, -1):
            m.ctx.vg[0, i] += sgn * h
            d.append((g * m.bands(K, nband)).sum())
            m.ctx.vg[0, i] -= sgn * h
        want[0, i] = (d[0] - d[1]) / (2 * h)
    assert np.abs(got - want).max() < 1e-9 * np.abs(want).max()
    last = nk - (nk - 1) // 8 * 8
    assert vectors <= nk * nband + last * max(0, nvalence + 1 - nband) + max(nband, nvalence + 1)


@pytest.mark.parametrize("nk", [64, 100000])
def test_levels_asked_for(nk):
    m = autograd.BandModel.__new__(autograd.BandModel)
    m.ctx, m.sys, m.refpoint, m.nvalence = _Solver(), types.SimpleNamespace(npw=50), np.zeros(3), 18
    K = np.random.default_rng(1).uniform(-0.5, 0.5, (nk, 3))
    off = m.ctx.ref_energy(m.refpoint, 18)
    m.ctx.levels = 0
    e = m.bands(K, 2)
    assert np.abs(e - m.ctx.bands(K, 2, off)).max() < 1e-12
    assert m.ctx.levels - 2 * nk <= 2 * nk + 65536 + 19
