"""The gradient of chi over more k-points than one batch holds (2048 for small
bases) is the sum of the gradients over parts of the grid.  Bar: 1e-9 of the
largest component, the rounding of sums of this length in FP64 with a wide
margin (2100 terms, 1e-16 each, and the eigenvalues' own 1e-13)."""
import numpy as np
import pytest

from picomax_amd import capi

pytestmark = pytest.mark.gpu

VG = [3, 4, 8, 11, -0.1407, 0.05, 0.0, 0.0577, -0.2807, -0.05, 0.0, 0.0277]


@pytest.mark.parametrize("nk,parts", [(2100, (0, 700, 1400, 2100)), (513, (0, 512, 513)), (1, (0, 1))])
def test_batches_add_up(nk, parts):
    args = ["-crystal", "zb", "-a", "5.65", "-vg", ",".join(map(str, VG)), "-gcut", repr(4.1 ** 0.5), "-neps", "3"]
    inp = capi.Input(args)
    ctx = capi.Context(0)
    ctx.set_system(inp.system(), inp)
    rng = np.random.default_rng(nk)
    K, KW = rng.uniform(-0.4, 0.4, (nk, 3)), rng.uniform(0.5, 1.0, nk) / nk
    Q, nf = [[0.01, 0.002, 0.0]], 40
    off = ctx.ref_energy((0, 0, 0), 8)
    gre, gim = rng.normal(size=(2, 9 * 6 * nf))
    grad = lambda i, j: np.asarray(ctx.grad_chi(K[i:j], KW[i:j], Q, 20, off, 0, 0.2, nf, 0.3, gre, gim, kk=1))
    whole = grad(0, nk)
    summed = sum(grad(i, j) for i, j in zip(parts, parts[1:]))
    assert np.abs(whole).max() > 0
    assert np.abs(whole - summed).max() < 1e-9 * np.abs(whole).max()
    ctx.close()
