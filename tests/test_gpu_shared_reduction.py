"""Tridiagonalisation of a large matrix by 2, 4 and 8 workgroups, alone and after a round of one workgroup a
matrix, with the waits as they are and with a limit of no polls (PMX_WIDE_SPINS=0): there nearly every wait
ends before the other workgroups have published, and the matrices are reduced again.

Eigenvalues are held to numpy's on the oracle's H(k), 1e-10 eV, and the pairs' residuals to 1e-12 of ||H||,
the bars of the large bases elsewhere."""
import numpy as np
import pytest

import orc
from picomax_amd import capi

pytestmark = pytest.mark.gpu

TE_VG = [0.565323, 1.333333, 1.898656, 2.261292, 3.594626, 4.0] + [-0.2105, -0.1322, 0.0451, 0.0214, 0.0127, -0.0093] * 3
US = {0.565323: 0.0152, 1.333333: -0.0061, 1.898656: 0.0083}
UA = {0.565323: 0.0117, 1.333333: 0.0042, 1.898656: -0.0071}
SI_VG = [3, 4, 8, 11, -0.21, 0, 0.04, 0.08, -0.21, 0, 0.04, 0.08]


def _system(name, gcut2):
    gcut = gcut2 ** 0.5
    if name == "si":
        kw = dict(a=5.43, vg=SI_VG)
        args = ["-crystal", "zb", "-a", "5.43", "-vg", ",".join(map(str, SI_VG))]
    else:
        kw = dict(a=4.45, f=1.33, u=0.26, vg=TE_VG)
        args = ["-crystal", "te", "-a", "4.45", "-f", "1.33", "-u", "0.26", "-vg", ",".join(map(str, TE_VG))]
        if name == "te_so":
            kw.update(us_so=US, ua_so=UA)
            for opt, m in (("-us_so", US), ("-ua_so", UA)):
                args += [opt, ",".join("%r:%r" % x for x in m.items())]
    inp = capi.Input(args + ["-gcut", repr(gcut)])
    ctx = capi.Context(0)
    ctx.set_system(inp.system(), inp)
    return ctx, orc.System("zb" if name == "si" else "te", gcut=gcut, **kw)


# workgroups a matrix: 8, 4, 2, 2, 4 beside a full round of 256, and the real form's 8 and 2
@pytest.mark.parametrize("name,gcut2,nk", [("te_so", 9.0, 3), ("te", 9.6, 50), ("te", 9.6, 128), ("te_so", 9.0, 90),
                                           ("te", 10.6, 300), ("si", 36.0, 5), ("si", 36.0, 100)])
@pytest.mark.parametrize("spins", [None, "0"])
def test_shared_pairs(monkeypatch, name, gcut2, nk, spins):
    if spins is not None:
        monkeypatch.setenv("PMX_WIDE_SPINS", spins)
    ctx, s = _system(name, gcut2)
    K = np.random.default_rng(nk).uniform(-0.4, 0.4, (nk, 3))
    for _ in range(3):  # eager, captured, replayed
        ev, vec = ctx.eig(K, 16, vectors=True)
    low = ctx.bands(K, 16, 0.0)
    for k in {0, nk // 2, nk - 1}:
        H = s.hamiltonian(K[k])
        w = np.linalg.eigvalsh(H)
        z = vec[k].T
        assert np.abs(ev[k] - w[:16]).max() < 1e-10
        assert np.abs(low[k] - w[:16]).max() < 1e-10
        assert np.abs(H @ z - z * ev[k]).max() < 1e-12 * np.abs(w).max()
    ctx.close()
