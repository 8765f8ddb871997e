"""Band fits solve the reference point with the k-points: batches of every split against separate calls."""
import numpy as np
import pytest

from picomax_amd import autograd

pytestmark = pytest.mark.gpu

ARGS = ["-crystal", "zb", "-a", "5.65", "-gcut", repr(8.1 ** 0.5),
        "-vg", "3,4,8,11,-0.14,0.07,0.0277,0.0635,-0.28,-0.07,0.0277,0.0435"]


# k-points against a batch of four, fewer and more bands than valence states, no valence states, all states
@pytest.mark.parametrize("nk", [0, 1, 3, 4, 5, 8, 9])
@pytest.mark.parametrize("nband,nvalence", [(4, 8), (8, 8), (12, 8), (5, 1), (6, 0), (6, 54)])
def test_offset_in_the_batch(nk, nband, nvalence):
    m = autograd.BandModel(ARGS, refpoint=(0.1, 0.05, 0.0), nvalence=nvalence, batch=4)
    n2 = 2 * m.sys.npw
    r = np.random.default_rng(nk)
    K, g = r.uniform(-0.5, 0.5, (nk, 3)), r.normal(size=(nk, nband))
    want = m.ctx.bands(K, nband, m.offset())
    got = m.bands(K, nband)
    assert got.shape == want.shape and (nk == 0 or np.abs(got - want).max() < 1e-11)
    if nk == 0:
        return
    want = m.ctx.grad_bands(K, nband, g)
    if 0 < nvalence < n2:
        ref = np.zeros((1, nvalence + 1))
        ref[0, nvalence - 1:] = -0.5 * g.sum()
        want += m.ctx.grad_bands(m.refpoint[None, :], nvalence + 1, ref)
    assert np.abs(m.grad(K, nband, g) - want).max() < 1e-9 * np.abs(want).max()


def test_adjoint_buffers_between_calls():
    """Calls of several sizes on one context, larger and smaller in turn, against a context of their own."""
    r = np.random.default_rng(1)
    vary = [(12, 20, 2, 30), (3, 12, 1, 9), (12, 20, 2, 30), (20, 24, 1, 50), (1, 12, 3, 5), (20, 24, 1, 50)]
    m = autograd.BandModel(ARGS, nvalence=8)
    for nk, nband, nq, nfreq in vary:
        K, KW, Q = r.uniform(-0.5, 0.5, (nk, 3)), np.full(nk, 1.0 / nk), r.uniform(0.01, 0.1, (nq, 3))
        e = m.ctx.bands(np.concatenate([K] + [K + q for q in Q]), nband, 0.0)
        a = (K, KW, Q, nband, (e[:, 0].max() + e[:, nband - 1].min()) / 2, 1, 0.3, nfreq, 0.2)
        g, gre, gim = (r.normal(size=n) for n in ((nk, nband), 9 * nq * nfreq, 9 * nq * nfreq))
        own = autograd.BandModel(ARGS, nvalence=8)
        for f in (lambda c: c.grad_bands(K, nband, g), lambda c: c.grad_chi(*a, gre, gim, kk=1)):
            want = f(own.ctx)
            for _ in range(3):
                assert np.abs(f(m.ctx) - want).max() < 1e-9 * np.abs(want).max()
