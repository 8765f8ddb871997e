"""Device memory that a context holds between gradients of chi."""
import numpy as np
import pytest
import torch

from picomax_amd import capi

pytestmark = pytest.mark.gpu

ARGS = ["-crystal", "zb", "-a", "5.65", "-gcut", repr(19.0 ** 0.5), "-neps", "59",
        "-vg", "3,4,8,11,-0.14,0.07,0.0277,0.0635,-0.28,-0.07,0.0277,0.0435"]


# a call whose buffers are kept, and one whose overlaps alone (4 x 14 transitions, 177 components, twice, 16 bytes)
# take 0.65 GB, with 0.52 GB of eigenvectors and 0.16 GB of their gradients
@pytest.mark.parametrize("nk", [20, 2048])
def test_held_memory(nk):
    """At most 1 GiB beside what the eigensolver keeps for a batch: 40 N^2 bytes a matrix (scratch 32, reflectors 8) and
    less than 2 N^2 for d, e and the like."""
    N = 89
    ctx = capi.Context(0)
    inp = capi.Input(ARGS)
    ctx.set_system(inp.system(), inp)
    r = np.random.default_rng(nk)
    K, Q = r.uniform(-0.4, 0.4, (nk, 3)), [[0.01, 0.0, 0.0]]
    off = ctx.ref_energy((0, 0, 0), 8)
    nfreq = 8
    n = 9 * 59 * 60 // 2 * nfreq
    g = np.zeros(n)
    g[:nfreq] = 1.0  # the head element only
    a = (K, np.full(nk, 1.0 / nk), Q, 36, off, 1, 0.3, nfreq, 0.5, g, g)
    ctx.bands(K[:20], 8)  # the library's own allocations
    free = torch.cuda.mem_get_info()[0]
    first = ctx.grad_chi(*a)
    held = free - torch.cuda.mem_get_info()[0]
    assert held < (1 << 30) + 42 * N * N * nk + (64 << 20), held
    again = ctx.grad_chi(*a)
    assert np.abs(again - first).max() < 1e-9 * np.abs(first).max()
    ctx.close()
