"""Adjoint sums: workspaces smaller than the query's answer."""

import ctypes
import sys

import numpy as np
import pytest
import torch

from gstools_amd import _native

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _case(d, n, p, seed):
    rs = np.random.RandomState(seed)
    arrays = (rs.normal(size=(d, n)) * 0.3, rs.normal(size=n), rs.normal(size=n), rs.uniform(-20.0, 20.0, (d, p)),
              rs.normal(size=p))
    return [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in arrays]


def _adjoint(args, precision, ws_bytes):
    """Status and gradients of one call with a workspace of ws_bytes."""
    cov, z1, z2, pos, g = args
    d, n = cov.shape
    g = g if precision == "fp64" else g.float()
    out = [torch.full(s, float("nan"), dtype=torch.float64, device="cuda") for s in ((n,), (n,), (d, n))]
    ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device="cuda")
    lib = _native.lib()
    fn = lib.gsx_summate_adjoint_f64 if precision == "fp64" else lib.gsx_summate_adjoint_f32
    st = fn(d, n, pos.shape[1], _ptr(cov), _ptr(z1), _ptr(z2), _ptr(pos), _ptr(g), *(_ptr(o) for o in out), _ptr(ws),
            ws_bytes, None)
    torch.cuda.synchronize()
    return st, out


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("d,n,p,chunks", [(2, 300, 2000, 8), (3, 2048, 100_000, 196), (1, 100, 65, 1),
                                          (2, 20_000, 9000, 18),
                                          (1, 10_000, 13_312, 51)])
def test_adjoint_takes_the_least_workspace(d, n, p, chunks, precision):
    """chunks: ceil(s / ceil(s / m)) of the header, or the query's number (last case).
    The float64 entry needs the query's answer."""
    _say(f"adjoint workspace d={d} N={n} P={p} {precision}")
    args = _case(d, n, p, n + p)
    most = int(_native.lib().gsx_summate_adjoint_workspace(d, n, p))
    least = (2 + 2 * d) * n * chunks * 8
    assert least <= most
    if precision == "fp64":
        least = most
    st, want = _adjoint(args, precision, most)
    assert st == 0
    st, got = _adjoint(args, precision, least)
    assert st == 0
    assert _adjoint(args, precision, least - 1)[0] == -4  # GSX_E_WORKSPACE
    # the float64 sums in another grouping, P |g x| 2^-53 each way, |z| < 8; the FP32 partial
    # sums over 256 points are the same whatever the chunks
    bound = 2.0 * p * 2.0**-53 * float(args[4].abs().sum()) * 20.0 * 8.0 * 2.0
    for a, b in zip(got, want):
        assert bool(torch.isfinite(a).all()) and float((a - b).abs().max()) <= bound
