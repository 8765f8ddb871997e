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
