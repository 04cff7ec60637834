"""The streaming form of the equations (csrc/bssn_rhs_stream.h, what the FP64
kernels run) built on the host against the reference's own generated equations
(tests/golden/algebra_points*.npz): the standard gauge with two parameter
sets, and its gauge instantiation on every other build. The bound is the one
the generated headers are held to on the same vectors (tests/test_abi.py)."""
import ctypes as C
import os

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
GOLD = os.path.join(ROOT, "tests", "golden")


def stream_points(inp, lam, lamf, xi=(0, 0, 0), gauge=0, rochester=0, ssl=0, t=0.0):
    dp = C.POINTER(C.c_double)
    f = C.CDLL(os.path.join(ROOT, "dendro-gr_amd", "lib", "libdgr_algebra_host.so")).dgr_host_bssn_stream
    f.argtypes = [dp, C.c_int64, dp, dp, dp, C.c_int, C.c_int, C.c_int, C.c_double, dp]
    out = np.full((len(inp), 24), np.nan)
    arrays = [np.array(list(v), float) for v in (lam, lamf, xi)]
    rc = f(inp.ctypes.data_as(dp), len(inp), *[a.ctypes.data_as(dp) for a in arrays], gauge, rochester, ssl, t,
           out.ctypes.data_as(dp))
    assert rc == 0, "the phases did not run in the order of kStreamVar"
    return out


@pytest.mark.parametrize("gauge", [0, 1])
@pytest.mark.parametrize("pset", ["A", "B"])
def test_standard_gauge(pset, gauge):
    g = np.load(os.path.join(GOLD, "algebra_points.npz"))
    lam, lf = {"A": ((1, 1, 1, 1), (1.0, 0.0)), "B": ((2, 3, 5, 7), (0.7, 0.3))}[pset]
    out = stream_points(np.ascontiguousarray(g["inputs"]), lam, lf, gauge=gauge)
    ref = g[f"out_{pset}"]
    err = np.abs(out - ref).max(0) / np.abs(ref).max(0)
    assert err.max() < 1e-13, err


@pytest.mark.parametrize("name", ["rochester", "rochester_etafunc", "ssl", "ssl_etafunc", "rochester_ssl",
                                  "rochester_ssl_etafunc"])
def test_other_gauges(name):
    import oracle as O
    from test_oracle_golden import gauge_params
    inp = np.ascontiguousarray(np.load(os.path.join(GOLD, "algebra_points.npz"))["inputs"].copy())
    ref = np.load(os.path.join(GOLD, "algebra_points_gauge.npz"))[f"out_{name}"]
    p = gauge_params(name)
    if p.eta_func:
        inp[:, 162] = O.eta_func_points(inp, p)
    out = stream_points(inp, p.lambda_, p.lambda_f, p.xi, 1, p.rochester, p.ssl, p.time)
    live = np.abs(ref).max(0) > 0
    err = np.abs(out - ref).max(0)[live] / np.abs(ref).max(0)[live]
    assert err.max() < 1e-13, err
    np.testing.assert_array_equal(out[:, ~live], 0.0)
