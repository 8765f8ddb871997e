"""The per-transition sum (`direct`, triangle and rectangle broadening, the
principal value of chi_LL and chi_xyz): frequencies on both sides of its blocks
of 32, bases of less than one tile and of several, few transitions and many.

Against the FP64 oracle, 1e-8 of each slice's max (or of 1e-4 of the largest
value, for slices that vanish by symmetry), the bar of the chi fixtures; 1e-5
with the principal value, whose poles magnify the eigenvalues' last bits."""
import numpy as np
import pytest

import orc
from picomax_amd import capi, kpoints

pytestmark = pytest.mark.gpu

VG = [3, 4, 8, 11, -0.1407, 0.05, 0.0, 0.0577, -0.2807, -0.05, 0.0, 0.0277]


def _check(gcut2, neps, us, nk, nband, nfreq, delta, ll, kk):
    gcut = gcut2 ** 0.5
    args = ["-crystal", "zb", "-a", "5.43", "-vg", ",".join(map(str, VG)), "-gcut", repr(gcut), "-neps", str(neps)]
    if us:
        args += ["-us_so", ",".join("%r:%r" % kv for kv in us.items())]
    inp = capi.Input(args)
    ctx = capi.Context(0)
    ctx.set_system(inp.system(), inp)
    s = orc.System("zb", a=5.43, vg=VG, gcut=gcut, neps=neps, us_so=us)
    K = kpoints.gamma_grid("zb", nk) + np.array([0.013, 0.027, 0.041])
    KW = np.full(len(K), 1.0 / len(K))
    off = ctx.ref_energy((0, 0, 0), 8)
    a = (K, KW, [[0.01, 0.002, 0.003]], nband, off, delta, 0.2, nfreq, 12.0 / max(nfreq, 12), kk)
    got, want = ctx.chi(*a, precision="direct", ll=ll), s.chi(*a, ll=ll)
    top = max(np.abs(w).max() for w in want)
    for g, w in zip(got, want):
        g, w = g.reshape(-1, nfreq), w.reshape(-1, nfreq)
        scale = np.maximum(np.abs(w).max(1), 1e-4 * top)
        assert (np.abs(g - w).max(1) <= (1e-5 if ll and not kk else 1e-8) * scale).all()
    ctx.close()


@pytest.mark.parametrize("nfreq", [1, 31, 32, 33, 64, 97])
@pytest.mark.parametrize("delta", [0, 1, 2, 3])
def test_frequencies(delta, nfreq):
    _check(8.1, 3, None, 2, 24, nfreq, delta, 0, 0)


@pytest.mark.parametrize("neps", [1, 5, 6, 11])
@pytest.mark.parametrize("us", [None, {3: 0.01, 8: 0.005}])
@pytest.mark.parametrize("ll,kk", [(0, 1), (1, 0), (2, 0)])
def test_bases(neps, us, ll, kk):
    _check(4.1, neps, us, 2, 24, 40, 2 if ll == 0 else 0, ll, kk)


@pytest.mark.parametrize("nk,nband", [(1, 10), (1, 24), (3, 24)])
def test_transitions(nk, nband):
    _check(8.1, 3, None, nk, nband, 45, 2, 0, 0)
