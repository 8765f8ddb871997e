"""The operation count that the kernel timings give for eps_M: N^3 / 3 complex multiply-adds a matrix by elimination,
2 N^3 by the Gauss-Jordan inverse, eight operations each."""
import numpy as np
import pytest

from picomax_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("neps", [9, 130])
@pytest.mark.parametrize("call,count", [("epsM", 8 / 3), ("full", 16), ("macro", 16 / 3)])
def test_eps_counts(neps, call, count):
    inp = capi.Input(["-crystal", "zb", "-a", "5.43", "-vg", "3,4,8,11" + ",-0.21,0,0.04,0.08" * 2, "-gcut", "4.9",
                      "-neps", str(neps)])
    ctx = capi.Context(0)
    ctx.set_system(inp.system(), inp)
    nfreq, nblk = 3, neps * (neps + 1) // 2 * 3
    x = np.zeros(9 * nblk)
    ctx.profile(True)
    if call == "macro":
        ctx.eps_macro(x, x, [[0.01, 0.0, 0.0]], nfreq, 0.1)
    else:
        ctx.epsinv(x[:nblk], x[:nblk], 1, nfreq, full=call == "full")
    rep = ctx.profile_report()
    ctx.close()
    got = rep["epsinv"]["flops"]
    assert abs(got / (count * neps ** 3 * nfreq) - 1) < 1e-6, rep
