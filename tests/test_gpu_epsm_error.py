"""Rounding of eps_M from the elimination against that from the whole inverse, on the same dielectrics (a few hundred
damped oscillators): the rms relative error may not exceed the inverse's by more than a fifth; over the frequencies of
a case the ratio scatters by less than a tenth.  The reference is an elimination in extended precision."""
import numpy as np
import pytest

from picomax_amd import capi

pytestmark = pytest.mark.gpu


def _chi(neps, nfreq):
    r = np.random.default_rng(neps)
    ns = 4 * neps
    amp = (r.normal(size=(ns, neps)) + 1j * r.normal(size=(ns, neps))) / (1 + np.arange(neps) / 6.0)
    w0, w = r.uniform(3, 15, ns), np.linspace(0, 20, nfreq)
    osc = 60.0 / ns / (w0 ** 2 - w[:, None] ** 2 - 0.3j * w[:, None])
    m, n = np.tril_indices(neps)
    return m, n, (osc @ (amp[:, m] * amp[:, n].conj())).T  # [element][f]


# one and two rows a lane in registers, and the workspace form
@pytest.mark.parametrize("neps,nfreq", [(60, 400), (127, 150), (137, 150)])
def test_no_worse_than_inverse(neps, nfreq):
    m, n, x = _chi(neps, nfreq)
    ctx = capi.Context(0)
    inp = capi.Input(["-crystal", "zb", "-a", "5.43", "-vg", "3,4,8,11" + ",-0.21,0,0.04,0.08" * 2, "-gcut", "4.9",
                      "-neps", str(neps)])
    ctx.set_system(inp.system(), inp)
    a = (np.ascontiguousarray(x.real), np.ascontiguousarray(x.imag), 1, nfreq)
    got, other = ctx.epsinv(*a)[0][0], ctx.epsinv(*a, full=True)[0][0]
    ctx.close()
    E = np.zeros((nfreq, neps, neps), np.clongdouble)
    E[:, n, m], E[:, m, n] = x.conj().T, x.T
    E += np.eye(neps)
    B = np.concatenate([E[:, :, np.r_[1:neps, 0]], np.eye(neps)[None, :, :1].repeat(nfreq, 0)], 2)
    i = np.arange(nfreq)
    for k in range(neps - 1):
        p = k + np.abs(B[:, k:, k]).argmax(1)
        B[i, p], B[:, k] = B[:, k].copy(), B[i, p].copy()
        B[:, k + 1:, k:] -= (B[:, k + 1:, k] / B[:, k, k][:, None])[:, :, None] * B[:, None, k, k:]
    want = B[:, -1, -2] / B[:, -1, -1]
    rms = lambda e: float(np.sqrt((np.abs((e - want) / want) ** 2).mean()))  # noqa: E731
    assert rms(got) < 1.2 * rms(other), (rms(got), rms(other))
