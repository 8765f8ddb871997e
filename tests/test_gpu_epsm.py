"""eps_M and the loss function without the full inverse (Gaussian elimination
to the head element) against numpy's inverse, at sizes around a wave, the
largest that registers hold and the first that the workspace takes; and not-a-number
input, which ends as not-a-number.  1e-11 relative: eps x cond(eps) x a
modest constant for these matrices (condition numbers below 1e3)."""
import numpy as np
import pytest

from picomax_amd import capi

pytestmark = pytest.mark.gpu

VG = "3,4,8,11,-0.21,0,0.04,0.08,-0.21,0,0.04,0.08"


def _ctx(neps):
    inp = capi.Input(["-crystal", "zb", "-a", "5.43", "-vg", VG, "-gcut", "6.0", "-neps", str(neps)])
    ctx = capi.Context(0)
    ctx.set_system(inp.system(), inp)
    return ctx


@pytest.mark.parametrize("neps", [1, 2, 3, 4, 5, 15, 16, 31, 32, 59, 62, 63, 64, 65, 89, 126, 127, 128, 181, 259])
def test_epsm_against_numpy(neps):
    nq, nf = 2, 5
    rng = np.random.default_rng(neps)
    ne2 = neps * (neps + 1) // 2
    z = rng.normal(size=(nq, ne2, nf)) + 1j * rng.normal(size=(nq, ne2, nf))
    z *= 0.3 / np.sqrt(neps)
    m, n = np.tril_indices(neps)
    z[:, m == n] += 1.0 + np.arange(neps)[None, :, None] / neps
    ctx = _ctx(neps)
    eM, elf = ctx.epsinv(z.real, z.imag, nq, nf)
    E = np.zeros((nq, nf, neps, neps), complex)
    zt = z.transpose(0, 2, 1)
    E[..., n, m] = zt.conj()
    E[..., m, n] = zt
    E += np.eye(neps)
    assert np.linalg.cond(E).max() < 1e3
    g = np.linalg.inv(E)[..., 0, 0]
    assert np.abs(eM * g - 1).max() < 1e-11
    assert np.abs(elf + g.imag).max() < 1e-11 * np.abs(g).max()
    ctx.close()


@pytest.mark.parametrize("neps", [4, 97, 130])
def test_pivoting_and_nan(neps):
    """A zero leading diagonal (pivots must come from other rows) and one NaN."""
    ne2 = neps * (neps + 1) // 2
    m, n = np.tril_indices(neps)
    z = np.zeros((1, ne2, 2), complex)
    rng = np.random.default_rng(7)
    z[0, :, 0] = rng.normal(size=ne2) + 1j * rng.normal(size=ne2)
    z[0, m == n, 0] = -1.0  # eps diagonal 0
    z[0, :, 1] = z[0, :, 0]
    z[0, -2, 1] = np.nan
    ctx = _ctx(neps)
    eM, elf = ctx.epsinv(z.real, z.imag, 1, 2)
    E = np.zeros((neps, neps), complex)
    E[n, m] = z[0, :, 0].conj()
    E[m, n] = z[0, :, 0]
    E += np.eye(neps)
    g = np.linalg.inv(E)[0, 0]
    assert abs(eM[0, 0] * g - 1) < 1e-13 * np.linalg.cond(E) * neps
    assert np.isnan(eM[0, 1]) and np.isnan(elf[0, 1])
    ctx.close()
