"""The eigenvalue kernels that small batches take (several lanes per level),
and the economised broadening tables, each at the sizes where they change.

Eigenvalues are held to numpy's on the oracle's H(k), 1e-10 eV, the bar of the
band fixtures.  chi of the binned FP64 path is held to the per-transition sum
(`direct`) within 1e-8 of each slice's maximum, the bar of the chi fixtures
(both tables are cut below 1e-11 of the broadening's peak)."""
import numpy as np
import pytest

import orc
from picomax_amd import capi, kpoints

pytestmark = pytest.mark.gpu

VG = [3, 4, 8, 11, -0.21, 0, 0.04, 0.08, -0.21, 0, 0.04, 0.08]
VG_AB = [3, 4, 8, 11, -0.1407, 0.05, 0.0, 0.0577, -0.2807, -0.05, 0.0, 0.0277]


def _pair(vg, gcut2, neps=1, us=None):
    gcut = gcut2 ** 0.5
    args = ["-crystal", "zb", "-a", "5.43", "-vg", ",".join(map(str, vg)), "-gcut", repr(gcut), "-neps", str(neps)]
    if us:
        args += ["-us_so", ",".join("%r:%r" % kv for kv in us.items())]
    inp = capi.Input(args)
    ctx = capi.Context(0)
    ctx.set_system(inp.system(), inp)
    return ctx, orc.System("zb", a=5.43, vg=vg, gcut=gcut, neps=neps, us_so=us)


def _eig(s, k):
    return np.linalg.eigvalsh(s.hamiltonian(k))


# nk spans one lane per level to 64, N even and odd, one level and all of them
@pytest.mark.parametrize("nk", [1, 2, 37, 260, 1500, 9000])
@pytest.mark.parametrize("gcut2,nband,us", [(12.0, 16, None), (12.0, 1, None), (3.1, 18, None), (0.5, 2, None),
                                            (4.1, 30, {3: 0.01, 8: 0.005})])
def test_levels_of_small_batches(nk, gcut2, nband, us):
    ctx, s = _pair(VG, gcut2, us=us)
    rng = np.random.default_rng(nk + nband)
    K = rng.uniform(-0.5, 0.5, (nk, 3))
    ev = ctx.bands(K, nband)
    for k in {0, nk // 2, nk - 1}:
        w = _eig(s, K[k])[:nband]
        assert np.abs(ev[k, :len(w)] - w).max() < 1e-10, (nk, k)
    ctx.close()


@pytest.mark.parametrize("target", [1e-2, 1e-6, 0.0])
def test_level_at_zero(target):
    """A level whose magnitude is far below the rounding level of H."""
    ctx, s = _pair(VG, 12.0)
    lo, hi = 0.0, 0.9
    d = np.array([0.6, 0.64, 0.48])
    assert _eig(s, lo * d)[0] < 0 < _eig(s, hi * d)[0]
    for _ in range(60):
        mid = 0.5 * (lo + hi)
        lo, hi = (mid, hi) if _eig(s, mid * d)[0] < target else (lo, mid)
    K = np.array([hi * d] * 5)
    ev = ctx.bands(K, 8)
    assert np.abs(ev - _eig(s, K[0])[None, :8]).max() < 1e-10
    ctx.close()


# (df/2)/epsilon from nearly 0 to the largest the binned path takes, both broadenings
@pytest.mark.parametrize("delta,eps,df", [(0, 0.3, 0.02), (0, 0.1, 0.05), (0, 0.1, 0.115), (1, 0.3, 0.02),
                                          (1, 0.05, 0.02), (1, 0.15, 0.1), (1, 0.1, 0.055)])
def test_economised_tables(delta, eps, df):
    ctx, _ = _pair(VG_AB, 8.1, neps=3)
    K = kpoints.gamma_grid("zb", 3) + np.array([0.013, 0.027, 0.041])
    KW = np.full(len(K), 1.0 / len(K))
    off = ctx.ref_energy((0, 0, 0), 8)
    a = (K, KW, [[0.01, 0.0, 0.0]], 24, off, delta, eps, 120, df, 0)
    got, want = ctx.chi(*a, precision="fp64"), ctx.chi(*a, precision="direct")
    for g, w in zip(got, want):
        g, w = g.reshape(-1, 120), w.reshape(-1, 120)
        scale = np.maximum(np.abs(w).max(1), 1e-4 * np.abs(w).max())
        assert (np.abs(g - w).max(1) / scale).max() < 1e-8
    ctx.close()


TE = ["-crystal", "te", "-a", "4.45", "-f", "1.33", "-u", "0.26", "-vg",
      "0.565323,1.333333,1.898656,2.261292,3.594626,4.0" + ",-0.2105,-0.1322,0.0451,0.0214,0.0127,-0.0093" * 3]
TE_SO = ["-us_so", "0.565323:0.0152,1.333333:-0.0061,1.898656:0.0083",
         "-ua_so", "0.565323:0.0117,1.333333:0.0042,1.898656:-0.0071"]
SI = ["-crystal", "zb", "-a", "5.43", "-vg", ",".join(map(str, VG))]


# bases whose matrix lies in global memory: the smallest, sizes around multiples
# of 64 and 128 rows, complex, spinor and real, one matrix to more than one per CU
@pytest.mark.parametrize("args,gcut2,nk", [(TE, 9.0, 1), (TE, 9.6, 3), (TE, 16.0, 300), (TE + TE_SO, 5.0, 2),
                                           (TE + TE_SO, 9.0, 5), (TE + TE_SO, 16.0, 2), (TE + TE_SO, 20.0, 2),
                                           (SI, 36.0, 2), (SI, 48.0, 3)])
def test_vectors_of_large_bases(args, gcut2, nk):
    """Eigenvalues against numpy (1e-10 eV) and residuals of the pairs (1e-12 of ||H||): what the
    tridiagonalisation and its reflectors decide."""
    inp = capi.Input(args + ["-gcut", repr(gcut2 ** 0.5)])
    ctx = capi.Context(0)
    ctx.set_system(inp.system(), inp)
    d = dict(zip(args[::2], args[1::2]))
    maps = [{float(k): float(v) for k, v in (p.split(":") for p in d[o].split(","))} if o in d else None
            for o in ("-us_so", "-ua_so")]
    s = orc.System(d["-crystal"], a=float(d["-a"]), f=float(d["-f"]) if "-f" in d else None,
                   u=float(d["-u"]) if "-u" in d else None, vg=[float(x) for x in d["-vg"].split(",")],
                   gcut=gcut2 ** 0.5, us_so=maps[0], ua_so=maps[1])
    rng = np.random.default_rng(nk)
    K = rng.uniform(-0.4, 0.4, (nk, 3))
    ev, vec = ctx.eig(K, 24, vectors=True)
    for k in {0, nk - 1}:
        H = s.hamiltonian(K[k])
        w = np.linalg.eigvalsh(H)
        z = vec[k].T
        assert np.abs(ev[k] - w[:24]).max() < 1e-10
        assert np.abs(H @ z - z * ev[k]).max() < 1e-12 * np.abs(w).max()
    ctx.close()


# complex bases in LDS, on both sides of the size where the default changes
# (29 / 30) and around multiples of the 6 x 6 tile
@pytest.mark.parametrize("gcut2,us", [(0.5, {3: 0.01}), (3.1, {3: 0.01}), (4.1, {3: 0.01}), (8.1, None), (8.1, {3: 0.01}),
                                      (11.1, None), (11.1, {3: 0.01}), (19.1, None), (16.1, {3: 0.01})])
@pytest.mark.parametrize("nk", [1, 5])
def test_vectors_of_small_complex_bases(gcut2, us, nk):
    ctx, s = _pair(VG_AB, gcut2, us=us)
    K = np.random.default_rng(7).uniform(-0.5, 0.5, (nk, 3))
    n = s.hamiltonian(K[0]).shape[0] // (1 if us else 2)
    nb = min(n, 12) if us else 2 * min(n, 12)
    ev, vec = ctx.eig(K, nb, vectors=True)
    for k in range(nk):
        H = s.hamiltonian(K[k])
        V = vec[k].T
        assert np.abs(ev[k] - np.linalg.eigvalsh(H)[:nb]).max() < 1e-10
        assert np.abs(H @ V - V * ev[k]).max() < 1e-9
    ctx.close()


# large bases shared by 2, 4 and 8 workgroups, and the rest of a batch that fills
# the GPU once; last panels of 1 to 4 columns, one and two rows a thread
@pytest.mark.parametrize("args,gcut2,nk", [(TE, 9.6, 128), (TE, 16.0, 64), (TE + TE_SO, 9.0, 33), (TE + TE_SO, 16.0, 100),
                                           (TE + TE_SO, 16.0, 40), (TE, 10.6, 257), (SI, 36.0, 90), (SI, 48.0, 60),
                                           (SI, 80.0, 7)])
def test_shared_large_bases(args, gcut2, nk):
    """Eigenvalues against one matrix per call (1e-10 eV), which the test above holds to numpy; orthonormal vectors."""
    ctx = capi.Context(0)
    inp = capi.Input(args + ["-gcut", repr(gcut2 ** 0.5)])
    ctx.set_system(inp.system(), inp)
    K = np.random.default_rng(nk).uniform(-0.4, 0.4, (nk, 3))
    ev, vec = ctx.eig(K, 20, vectors=True)
    for k in range(0, nk, max(1, nk // 5)):
        one, _ = ctx.eig(K[k:k + 1], 20, vectors=True)
        assert np.abs(ev[k] - one[0]).max() < 1e-10
    for k in (0, nk - 1):
        z = vec[k]
        assert np.abs(z.conj() @ z.T - np.eye(len(z))).max() < 1e-10
    ctx.close()


# bases in global memory, q in one batch with k: all at once, in groups (100 k:
# four q at a time), with and without a captured step, the smallest counts
@pytest.mark.parametrize("nk,nq", [(1, 2), (3, 3), (8, 7), (100, 3), (100, 4), (100, 6), (100, 9), (170, 2), (171, 3), (260, 2)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_q_batches(nk, nq, precision):
    """A list of q against one q per call: the same products in the same order, up to the eigensolver's rounding."""
    ctx = capi.Context(0)
    inp = capi.Input(TE + ["-gcut", repr(9.6 ** 0.5), "-neps", "3"])
    ctx.set_system(inp.system(), inp)
    K = np.random.default_rng(nk).uniform(-0.4, 0.4, (nk, 3))
    KW = np.full(nk, 1.0 / nk)
    Q = np.array([[0.0, 0.0, 0.03 * (i + 1)] for i in range(nq)])
    e = ctx.bands(np.concatenate([K] + [K + q for q in Q]), 24, 0.0)
    off = (e[:, 0].max() + e[:, 23].min()) / 2  # states on both sides of it at every point
    a = (24, off, 1, 0.1, 60, 0.1, 1)
    for _ in range(2):
        got = ctx.chi(K, KW, Q, *a, precision=precision)
        one = [ctx.chi(K, KW, q[None, :], *a, precision=precision) for q in Q]
        for i in (0, 1):
            g = got[i].reshape(9, nq, -1)
            w = np.stack([o[i].reshape(9, -1) for o in one], 1)
            assert np.abs(g - w).max() < (1e-10 if precision == "fp64" else 1e-5) * np.abs(w).max()
    ctx.close()


# bases below, at and above 16 states a tile, and one of two chunks of states (N > 224)
@pytest.mark.parametrize("args,gcut2,nband", [(SI, 3.1, 12), (SI, 8.1, 20), (SI, 12.0, 34), (TE, 13.6, 20), (TE + TE_SO, 9.0, 20)])
def test_chi_gradient_over_bases(args, gcut2, nband):
    """Directional derivative of a chi functional against central differences: h = 1e-5 Ry, truncation and
    rounding together below 1e-5 of the gradient's scale."""
    ctx = capi.Context(0)
    inp = capi.Input(args + ["-gcut", repr(gcut2 ** 0.5), "-neps", "2"])
    sysm = inp.system()
    ctx.set_system(sysm, inp)
    v0 = np.ctypeslib.as_array(sysm.vg, shape=(sysm.natom, sysm.nv)).copy()
    K = np.array([[0.11, 0.07, 0.19], [0.23, -0.05, 0.31]])
    Q = [[0.02, 0.01, 0.03]]
    e = ctx.bands(np.concatenate([K, K + Q[0]]), nband, 0.0)
    n = 2 * (np.argmax((e[:, 2::2].min(0) - e[:, 1:-2:2].max(0))) + 1)
    off = (e[:, n].min() + e[:, n - 1].max()) / 2
    a = (K, [0.5, 0.5], Q, nband, off, 1, 0.5, 40, 0.25)
    r = np.random.default_rng(3)
    re, im = ctx.chi(*a, kk=1)
    gr, gi = r.normal(size=re.shape), r.normal(size=im.shape)
    g = ctx.grad_chi(*a, gr, gi, kk=1)
    dv, h = r.normal(size=v0.shape), 1e-5
    f = []
    for sgn in (1, -1):
        ctx.set_form_factors(v0 + sgn * h * dv)
        x, y = ctx.chi(*a, kk=1)
        f.append((gr * x + gi * y).sum())
    ctx.close()
    assert abs((f[0] - f[1]) / (2 * h) - (g * dv).sum()) < 1e-5 * np.abs(g * dv).sum()
