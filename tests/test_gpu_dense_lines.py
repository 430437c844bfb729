"""Line calls of FMM plans of N <= 2048 as the tiled dense product on FP64 MFMA
(k_lines_gemm).  Sampled lines against the oracle, tolerance 1e-14 log2 N per line as in the other line
tests."""
import math

import numpy as np
import pytest

from conftest import announce, relerr

pytestmark = pytest.mark.gpu


def tol(n):
    return 1e-14 * math.log2(max(n, 2))


def run_lines(amd, plan, x, direction, strided, pad=0):
    """Every row of x (lines, N) in one call: back to back at distance N + pad,
    or (strided) with the lines interleaved, B + pad elements apart; the
    elements between stay untouched."""
    B, N = x.shape
    if strided:
        buf = np.zeros((N, B + pad))
        buf[:, :B] = x.T
        m = (B, 1, 0, B + pad)
    else:
        buf = np.zeros((B, N + pad))
        buf[:, :N] = x
        m = (B, N + pad, 0, 1)
    din, dout = amd.DeviceBuffer(buf.size), amd.DeviceBuffer(buf.size)
    din.upload(buf.ravel())
    dout.upload(np.full(buf.size, 7.0))
    plan.execute_lines_device(din.ptr, dout.ptr, direction, B, *m)
    plan.synchronize()
    y = dout.download().reshape(buf.shape)
    if pad:
        assert np.all(y[:, (B if strided else N):] == 7.0)
    return np.ascontiguousarray(y[:, :B].T) if strided else y[:, :N]


def check(orc, x, y, direction, maxs, rows):
    N = x.shape[1]
    op = orc.FMMPlan(N, maxs, 18, orc.BOTH)
    for r in rows:
        assert relerr(y[r], op.execute(np.ascontiguousarray(x[r]), direction)) <= tol(N), (r, direction)


@pytest.mark.parametrize("N,B", [(257, 2), (500, 33), (769, 40), (1000, 65), (1536, 17),
                                 (1537, 127), (1537, 128), (2047, 130), (2048, 128), (2049, 130)])
@pytest.mark.parametrize("strided", [False, True])
def test_fmm_plan_lines(amd, orc, monkeypatch, N, B, strided):
    """Line calls of FMM plans: the dense product up to N = 1536, from 128
    lines on up to 2048, the FMM past that; against the oracle and the FMM
    route (L2C_DENSE_MAXN=0)."""
    announce(f"FMM plan lines N={N} B={B} strided={strided}")
    monkeypatch.delenv("L2C_DIRECT_MAXN", raising=False)
    monkeypatch.setenv("L2C_DIRECT_LINES", "0")
    dense = N <= 1536 or (N <= 2048 and B >= 128)
    plan = amd.FMMPlan(N, 64, 18, 2)
    assert plan.info()["L"] >= 1
    monkeypatch.setenv("L2C_DENSE_MAXN", "0")
    fmm = amd.FMMPlan(N, 64, 18, 2)
    x = np.random.default_rng(N + B).uniform(-1, 1, (B, N)) / np.sqrt(np.arange(1, N + 1))
    for d in (0, 1):
        plan.profile(True)
        y = run_lines(amd, plan, x, d, strided, pad=1)
        assert (set(plan.profile_read()) == {"k_direct"}) == dense
        plan.profile(False)
        check(orc, x, y, d, 64, [0, B // 2, B - 1])
        z = run_lines(amd, fmm, x, d, strided, pad=1)
        assert max(relerr(y[r], z[r]) for r in range(B)) <= tol(N)
