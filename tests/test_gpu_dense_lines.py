"""Line calls as dense products on FP64 MFMA: k_lines_dense (direct plans of
N <= 256, more than 4,096 lines, or N <= 32) and k_lines_gemm (longer lines
and smaller calls, and the line calls of FMM plans of N <= 2048).  Sampled
lines against the oracle, tolerance 1e-14 log2 N per line as in the other line
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


# row tiles 1, 2 | 3, 4 | 5 .. 8 of the three widths, full and partly empty,
# odd lengths; 4,097 lines: past the tiled product's share, one line in the
# last tile; 70 lines: fewer tiles than the GPU holds
@pytest.mark.parametrize("N", [2, 15, 31, 32, 33, 63, 64, 65, 97, 128, 129, 191, 225, 255, 256])
@pytest.mark.parametrize("strided", [False, True])
@pytest.mark.parametrize("direction", [0, 1])
def test_whole_lines(amd, orc, N, strided, direction):
    B = 70 if N <= 32 else 4097
    announce(f"whole lines N={N} B={B} strided={strided} dir={direction}")
    x = np.random.default_rng(N).uniform(-1, 1, (B, N))
    plan = amd.FMMPlan(N, 64, 18, direction)
    y = run_lines(amd, plan, x, direction, strided, pad=3)
    check(orc, x, y, direction, 64, [0, 15, 16, 31, 32, B // 2, B - 2, B - 1])


def test_whole_lines_many_tiles(amd, orc):
    """60,001 lines: every work-group walks several tiles, some one more than
    others, the last tile holds one line."""
    for N, strided in ((256, False), (256, True), (100, False), (100, True), (40, True)):
        announce(f"whole lines N={N} B=60001 strided={strided}")
        x = np.random.default_rng(N).uniform(-1, 1, (60001, N))
        plan = amd.FMMPlan(N, 64, 18, 0)
        y = run_lines(amd, plan, x, 0, strided)
        check(orc, x, y, 0, 64, [0, 1, 31, 32, 24575, 24576, 49151, 49152, 59999, 60000])


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


@pytest.mark.parametrize("N,B", [(300, 40), (1000, 70), (1536, 33), (2048, 130)])
@pytest.mark.parametrize("direction", [0, 1])
def test_not_finite(amd, monkeypatch, N, B, direction):
    """A NaN or Inf on the FMM plans' dense route reaches the rows of its line
    and parity at or before its place, all of them, and no other."""
    announce(f"dense route, not finite N={N} B={B} dir={direction}")
    monkeypatch.setenv("L2C_DIRECT_LINES", "0")
    plan = amd.FMMPlan(N, 64, 18, direction)
    for strided in (False, True):
        for pos in (0, 1, 30, 31, 32, 33, N // 2, N // 2 + 17, N - 2, N - 1):
            for val in (np.inf, -np.inf, np.nan):
                x = np.random.default_rng(N).uniform(0.5, 1, (B, N))
                x[B // 2, pos] = val
                y = run_lines(amd, plan, x, direction, strided)
                want = np.zeros((B, N), bool)
                want[B // 2, pos % 2:pos + 1:2] = True
                assert np.array_equal(~np.isfinite(y), want), (strided, pos, val)


@pytest.mark.parametrize("N,maxs", [(200, 64), (1000, 64), (1201, 36)])
def test_blocks_of_planned_directions(amd, monkeypatch, N, maxs):
    """The parity blocks of a plan of one direction and of both, direct plans and FMM
    plans: the same results bit for bit, and no results in a direction not planned."""
    announce(f"dense blocks by direction N={N} maxs={maxs}")
    monkeypatch.delenv("L2C_DIRECT_MAXN", raising=False)
    monkeypatch.setenv("L2C_DIRECT_LINES", "0")
    x = np.random.default_rng(N).uniform(-1, 1, (50, N))
    both = amd.FMMPlan(N, maxs, 18, amd.BOTH)
    for d in (0, 1):
        one = amd.FMMPlan(N, maxs, 18, d)
        assert np.array_equal(run_lines(amd, one, x, d, False), run_lines(amd, both, x, d, False))
        with pytest.raises(amd.L2CError):
            run_lines(amd, one, x, 1 - d, False)


@pytest.mark.parametrize("N,B", [(40, 9), (200, 50), (256, 70), (300, 40), (1000, 70), (1536, 33),
                                 (2048, 130)])
@pytest.mark.parametrize("direction", [0, 1])
def test_tiled_product_not_finite(amd, monkeypatch, N, B, direction):
    """A NaN or Inf in a line that runs on the tiled dense product (direct plans and the
    FMM plans' dense route, the small-N routes on) reaches the rows of its line and
    parity at or before its place, all of them, and no other."""
    announce(f"tiled product, not finite N={N} B={B} dir={direction}")
    monkeypatch.delenv("L2C_DIRECT_MAXN", raising=False)
    monkeypatch.setenv("L2C_DIRECT_LINES", "0")
    plan = amd.FMMPlan(N, 64, 18, direction)
    plan.profile(True)
    for strided in (False, True):
        for pos in (0, 1, 15, 16, 30, 31, 32, 33, N // 2, N // 2 + 17, N - 2, N - 1):
            for val in (np.inf, -np.inf, np.nan):
                x = np.random.default_rng(N).uniform(0.5, 1, (B, N))
                x[B // 2, pos] = val
                y = run_lines(amd, plan, x, direction, strided)
                want = np.zeros((B, N), bool)
                want[B // 2, pos % 2:pos + 1:2] = True
                assert np.array_equal(~np.isfinite(y), want), (strided, pos, val)
    assert set(plan.profile_read()) == {"k_direct"}
