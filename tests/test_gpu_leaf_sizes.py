"""The FMM passes of plans with M = 18 at every leaf size s <= 64 (k_up with
the near-field band's work-groups beside it, k_far; k_band alone for directM
and the split pass): every remainder of s against the tiles of 16 rows and
columns, the vectors of two and the LDS layouts by s mod 4, with the last leaf
chunk full, one row short and nearly empty.  Against the oracle (the same FMM,
1e-14 log2 N as in the other transform tests) and the general downward kernel
(L2C_DOWN8=0)."""
import math

import numpy as np
import pytest

from conftest import announce, relerr

pytestmark = pytest.mark.gpu


def tol(n):
    return 1e-14 * math.log2(max(n, 2))


def lines(amd, plan, x, direction, strided, pad=0):
    """Every row of x (lines, N) in one call, back to back or interleaved; the
    elements between stay untouched."""
    B, N = x.shape
    buf = np.zeros((N, B + pad) if strided else (B, N + pad))
    if strided:
        buf[:, :B] = x.T
    else:
        buf[:, :N] = x
    din, dout = amd.DeviceBuffer(buf.size), amd.DeviceBuffer(buf.size)
    din.upload(buf.ravel())
    dout.upload(np.full(buf.size, 7.0))
    m = (B, 1, 0, B + pad) if strided else (B, N + pad, 0, 1)
    plan.execute_lines_device(din.ptr, dout.ptr, direction, B, *m)
    plan.synchronize()
    y = dout.download().reshape(buf.shape)
    if pad:
        assert np.all(y[:, (B if strided else N):] == 7.0)
    return np.ascontiguousarray(y[:, :B].T) if strided else y[:, :N]


@pytest.mark.parametrize("s", range(1, 65))
def test_leaf_size(amd, orc, monkeypatch, s):
    announce(f"leaf size {s}")
    for L, r in ((1, 0), (2, 7), (4, 1), (5, 64)):
        N = s * (4 << L) - min(r, (4 << L) - 1)
        if s == 1:
            N = 4 << L
        plan = amd.FMMPlan(N, s, 18, 2)
        info = plan.info()
        assert (info["s"], info["L"]) == (s, L)
        monkeypatch.setenv("L2C_DOWN8", "0")
        gen = amd.FMMPlan(N, s, 18, 2)
        monkeypatch.delenv("L2C_DOWN8")
        op = orc.FMMPlan(N, s, 18, 2)
        x = np.random.default_rng(64 * L + s).uniform(-1, 1, (3, N))
        for d in (0, 1):
            o = op.execute(np.ascontiguousarray(x[0]), d)
            y = plan.execute(x[0], d)
            assert relerr(y, o) <= tol(N), (N, d)
            assert relerr(y, gen.execute(x[0], d)) <= tol(N), (N, d)
            for strided in (False, True):
                z = lines(amd, plan, x, d, strided, pad=1)
                assert relerr(z[0], o) <= tol(N), (N, d, strided)
                o2 = op.execute(np.ascontiguousarray(x[2]), d)
                assert relerr(z[2], o2) <= tol(N), (N, d, strided)


@pytest.mark.parametrize("s,L", [(1, 5), (17, 3), (31, 4), (33, 3), (36, 8), (50, 9), (63, 4)])
@pytest.mark.parametrize("lagrange,precompute", [(0, 1), (1, 0)])
def test_leaf_variants(amd, orc, monkeypatch, s, L, lagrange, precompute):
    """Lagrange basis, the precomputed C2L band, strides, the split pass and
    the M2L's precision forms 1 and 2 at leaf sizes that are no multiple of 16."""
    N = s * (4 << L) - (3 if s > 1 else 0)
    announce(f"leaf size {s} N={N} lagrange={lagrange} precompute={precompute}")
    plan = amd.FMMPlan(N, s, 18, 2, lagrange, precompute)
    assert plan.info()["s"] == s
    op = orc.FMMPlan(N, s, 18, 2, lagrange, precompute)
    monkeypatch.setenv("L2C_DOWN_SPLIT", "1")
    split = amd.FMMPlan(N, s, 18, 2, lagrange, precompute)
    u = np.random.default_rng(s).uniform(-1, 1, N)
    for d in (0, 1):
        o = op.execute(u, d)
        y = plan.execute(u, d)
        assert relerr(y, o) <= tol(N)
        assert relerr(split.execute(u, d), y) <= tol(N)
        for form in (1, 2):
            plan.set_precision(form)
            assert relerr(plan.execute(u, d), o) <= 1e-13, form
        plan.set_precision(0)


@pytest.mark.parametrize("s", [5, 16, 18, 31, 32, 44, 64])
def test_band_alone(amd, orc, s):
    """directM (the near field alone), and unit vectors across the first and
    last leaf chunks, each seen by the near field and a block or two."""
    N = 64 * s - 5
    announce(f"band alone s={s}")
    plan = amd.FMMPlan(N, s, 18, 2)
    assert plan.info()["s"] == s
    op = orc.FMMPlan(N, s, 18, 2)
    u = np.random.default_rng(s).uniform(-1, 1, N)
    o = np.zeros(N)
    orc.lib().orc_directM(orc._p(u), orc._p(o), op._p, 1)
    assert relerr(plan.directM(u), o) <= tol(N)
    for d in (0, 1):
        for c in list(range(0, 4 * s, 7)) + list(range(N - 4 * s, N, 7)):
            u = np.zeros(N)
            u[c] = 1.0
            assert relerr(plan.execute(u, d), op.execute(u, d)) <= tol(N), (d, c)


@pytest.mark.parametrize("N,maxs,M", [(1000, 16, 10), (4000, 32, 20), (16284, 64, 24)])
def test_other_ranks(amd, orc, monkeypatch, N, maxs, M):
    """Ranks without kernels of their own: k_down8r, k_down8 and k_down."""
    announce(f"rank {M} N={N} maxs={maxs}")
    for name, value in (("L2C_DOWN_ROLES", "1"), ("L2C_DOWN_ROLES", "0"), ("L2C_DOWN8", "0")):
        monkeypatch.setenv(name, value)
        plan = amd.FMMPlan(N, maxs, M, 2)
        monkeypatch.delenv(name)
        op = orc.FMMPlan(N, maxs, M, 2)
        u = np.random.default_rng(N).uniform(-1, 1, N)
        for d in (0, 1):
            assert relerr(plan.execute(u, d), op.execute(u, d)) <= tol(N), (name, value, d)


@pytest.mark.parametrize("s", range(1, 65))
def test_many_lines(amd, orc, s):
    """Calls of many lines, whose band takes 8 chunks per work-group (the first
    two) or 16 (the last) for s > 32, contiguous and strided."""
    announce(f"many lines, leaf size {s}")
    for L, r, B in ((1, 0, 16), (3, 5, 37), (4, 1, 70)):
        N = 4 << L if s == 1 else s * (4 << L) - min(r, (4 << L) - 1)
        plan = amd.FMMPlan(N, s, 18, 2)
        assert plan.info()["s"] == s
        op = orc.FMMPlan(N, s, 18, 2)
        x = np.random.default_rng(64 * L + s).uniform(-1, 1, (B, N))
        for d in (0, 1):
            o = {l: op.execute(np.ascontiguousarray(x[l]), d) for l in (0, 7, 15, B - 1)}
            for strided in (False, True):
                z = lines(amd, plan, x, d, strided, pad=1)
                for l in o:
                    assert relerr(z[l], o[l]) <= tol(N), (N, d, strided, l)


@pytest.mark.parametrize("N,s,B", [(4096, 64, 20), (4000, 32, 17), (9000, 36, 33), (9000, 36, 3)])
@pytest.mark.parametrize("direction", [0, 1])
def test_not_finite(amd, N, s, B, direction):
    """A NaN or Inf reaches the rows of its own line that it belongs to, at or
    before its place and of its parity, and no other (the near field; upward
    of it the far field spreads it to all of them)."""
    announce(f"not finite N={N} B={B} dir={direction}")
    plan = amd.FMMPlan(N, s, 18, direction)
    for strided in (False, True):
        for pos in (0, 1, N // 3, N // 2 + 1, N - 130, N - 2, N - 1):
            for val in (np.inf, np.nan):
                x = np.random.default_rng(B).uniform(0.5, 1, (B, N))
                x[B // 2, pos] = val
                z = lines(amd, plan, x, direction, strided)
                want = np.zeros((B, N), bool)
                want[B // 2, pos % 2:pos + 1:2] = True
                bad = ~np.isfinite(z)
                assert not np.any(bad & ~want), (strided, pos, val)
                assert bad[B // 2, pos]
