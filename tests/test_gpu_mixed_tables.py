"""The binned chi of the mixed paths at every order count that their broadening tables take (3 to 12), against the
per-transition sum in FP64, by the measure and the bars of the chi fixtures: 1e-4 of each slice's maximum in FP32,
5e-3 in split BF16."""
import numpy as np
import pytest

import cli_args
from picomax_amd import capi, kpoints

pytestmark = pytest.mark.gpu

VG = "3,4,8,11,-0.1407,0.05,0.0,0.0577,-0.2807,-0.05,0.0,0.0277"


# (df/2)/epsilon 0.01 to 0.59 (Gaussian), 0.01 to 0.5 (Lorentzian)
@pytest.mark.parametrize("delta,eps,df", [(0, 1.0, 0.02), (0, 0.3, 0.02), (0, 0.1, 0.02), (0, 0.1, 0.03), (0, 0.1, 0.05),
                                          (0, 0.1, 0.08), (0, 0.1, 0.1), (0, 0.1, 0.118), (1, 1.0, 0.02), (1, 0.2, 0.02),
                                          (1, 0.1, 0.02), (1, 0.1, 0.03), (1, 0.05, 0.02), (1, 0.1, 0.06), (1, 0.1, 0.08),
                                          (1, 0.1, 0.1)])
@pytest.mark.parametrize("precision,bar", [("fp32", 1e-4), ("bf16x3", 5e-3)])
def test_orders(precision, bar, delta, eps, df):
    inp = capi.Input(["-crystal", "zb", "-a", "5.43", "-vg", VG, "-gcut", repr(8.1 ** 0.5), "-neps", "3"])
    ctx = capi.Context(0)
    ctx.set_system(inp.system(), inp)
    K = kpoints.gamma_grid("zb", 3) + np.array([0.013, 0.027, 0.041])
    a = (K, np.full(len(K), 1.0 / len(K)), [[0.01, 0.0, 0.0]], 24, ctx.ref_energy((0, 0, 0), 8), delta, eps, 120, df, 1)
    got, want = ctx.chi(*a, precision=precision), ctx.chi(*a, precision="direct")
    ctx.close()
    assert cli_args.slice_error(np.concatenate(got), np.concatenate(want), 9 * 6) < bar
