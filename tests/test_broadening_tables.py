"""The broadening's economised expansion over a frequency bin (picomax_amd/csrc/pmx_broadening.h, compiled here by
the host compiler) against the Taylor series it replaces: the rms error over a bin, at the offset where it is worst,
may not be larger, in FP64 and on the mixed paths.  A hundredth is left for the sampling of the bin."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include "pmx_broadening.h"
using namespace pmx;
/* out: rms errors of the Taylor series and of the economised one (of the peak), their orders */
extern "C" int table_errors(int delta, double eps, double df, double tol, double *out) {
    const int NT = taylor_order(delta, eps, df, tol);
    if (NT < 0) return 0;
    const Economised ec = economise(delta, eps, df, NT);
    const int Dm = int(6 * eps / df) + 2, W = 2 * Dm + 1, S = 400;
    std::vector<double> Kt, row(NT);
    kernel_table(delta, eps, df, -Dm, W, ec, Kt);
    const long double pi = 3.14159265358979323846264338L;
    auto exact = [&](long double x) {
        return delta == 1 ? eps / pi / (x * x + (long double)eps * eps)
                          : expl(-0.5L * x * x / ((long double)eps * eps)) / (eps * sqrtl(2 * pi));
    };
    long double worst[2] = {0, 0};
    for (int D = -Dm; D <= Dm; D++) {
        taylor_row(delta, eps, 0.5 * df, (D + 0.5) * df, NT, row.data());
        long double e[2] = {0, 0};
        for (int i = 0; i < S; i++) {
            const long double s = -1 + (2 * i + 1.0L) / S, want = exact((D + 0.5L + 0.5L * s) * df);
            long double p = 1, a = -want, b = -want;
            for (int n = 0; n < NT || n < ec.M; n++, p *= s) {
                if (n < NT) a += p * row[n];
                if (n < ec.M) b += p * Kt[(size_t)(D + Dm) * ec.M + n];
            }
            e[0] += a * a / S;
            e[1] += b * b / S;
        }
        for (int i = 0; i < 2; i++) worst[i] = std::max(worst[i], e[i]);
    }
    for (int i = 0; i < 2; i++) out[i] = (double)(sqrtl(worst[i]) / exact(0));
    out[2] = NT;
    out[3] = ec.M;
    return 1;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("tables")
    src, so = d / "t.cpp", d / "t.so"
    src.write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "picomax_amd", "csrc"),
                    "-o", str(so), str(src)], check=True)
    lib = ctypes.CDLL(str(so))
    lib.table_errors.argtypes = [ctypes.c_int] + [ctypes.c_double] * 3 + [ctypes.POINTER(ctypes.c_double)]
    return lib


# (df/2)/epsilon from nearly 0 to the largest the binned path takes; the truncations of FP64 and of the mixed paths
@pytest.mark.parametrize("delta", [0, 1])
@pytest.mark.parametrize("tol", [1e-11, 1e-6])
def test_no_worse_than_taylor(lib, delta, tol):
    eps, out = 0.1, (ctypes.c_double * 4)()
    tried = 0
    for r in np.concatenate([[0.01, 0.03], np.arange(0.05, 0.6, 0.0125)]):
        if not lib.table_errors(delta, eps, 2 * r * eps, tol, out):
            continue
        tried += 1
        taylor, econ, nt, m = out
        assert m <= nt
        # below 1e-14 of the peak both are rounding
        assert econ <= 1.01 * taylor + 1e-14, (r, taylor, econ, nt, m)
    assert tried > 10
