"""The device entry points on a caller's stream: torch tensors as the device
arrays and a torch.cuda.Stream as the stream, with torch work ordered before
and after the library's launches on that same stream (no host
synchronisation in between).  Results against the oracle."""
import math

import numpy as np
import pytest

from conftest import announce, relerr

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def test_execute_dct_and_batch_on_a_torch_stream(amd, orc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N = 1 << 16
    announce(f"torch stream N={N}")
    u = amd.coefficients(N, seed=21)
    plan = amd.FMMPlan(N, 64, 18, amd.BOTH)
    dct = amd.DCTPlan(N)
    bp = amd.BatchPlan([100, 3000, 512], 18, amd.L2C, tune=False)
    ub = amd.packed_coefficients([100, 3000, 512], seed=22)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        x = torch.zeros(N, dtype=torch.float64, device="cuda")
        y = torch.empty_like(x)
        v = torch.empty_like(x)
        xb = torch.zeros(ub.size, dtype=torch.float64, device="cuda")
        yb = torch.empty_like(xb)
        # the inputs are written by torch on s, then used by the library on s
        x.copy_(torch.from_numpy(u), non_blocking=False)
        x.mul_(2.0)
        xb.copy_(torch.from_numpy(ub))
        sp = s.cuda_stream
        plan.execute_device(x.data_ptr(), y.data_ptr(), amd.L2C, 1, sp)
        dct.execute_device(y.data_ptr(), v.data_ptr(), 3, sp)
        bp.execute_device(xb.data_ptr(), yb.data_ptr(), amd.L2C, sp)
        yb.mul_(0.5)  # torch work after the batch, same stream
        out_y, out_v, out_b = y.cpu(), v.cpu(), yb.cpu()
    s.synchronize()
    ref = orc.FMMPlan(N, 64, 18, orc.BOTH).execute(2 * u, 0)
    tol = 1e-14 * math.log2(N)
    assert relerr(out_y.numpy(), ref) < tol
    assert relerr(out_v.numpy(), orc.redft(ref, 3)) < 1e-15 * math.log2(2 * N) + tol
    off = 0
    for n in (100, 3000, 512):
        r = 0.5 * orc.FMMPlan(n, 64, 18, orc.BOTH).execute(ub[off:off + n], 0)
        assert relerr(out_b.numpy()[off:off + n], r) < 1e-14 * math.log2(n)
        off += n


def test_batch_graph_other_arrays(amd):
    """With the graph on: the first arrays that two calls in a row share are recorded and
    replayed; other arrays, the other direction and calls after l2c_batch_graph(0) run
    launch by launch, in turn with the replays, on the plan's and on a caller's stream;
    every result as without the graph, bit for bit."""
    announce("batch graph, other arrays")
    lengths = amd.log_uniform_lengths(300, seed=7)
    bp = amd.BatchPlan(lengths, 18, amd.BOTH, tune=False)
    u = [amd.packed_coefficients(lengths, seed=s) for s in (1, 2)]
    din = [amd.DeviceBuffer(bp.total) for _ in u]
    dout = [amd.DeviceBuffer(bp.total) for _ in u]
    for b, x in zip(din, u):
        b.upload(x)
    sp = torch.cuda.Stream().cuda_stream

    def call(k, d, stream=None):
        dout[k].upload(np.full(bp.total, 7.0))
        bp.execute_device(din[k].ptr, dout[k].ptr, d, stream=stream)
        torch.cuda.synchronize()
        return dout[k].download()

    ref = [[call(k, d) for d in (0, 1)] for k in (0, 1)]
    bp.graph(True)
    turns = [(0, 0)] * 3 + [(1, 0)] * 3 + [(0, 0), (1, 0)] * 3 + [(0, 1), (0, 0), (1, 1), (0, 0)]
    for stream in (None, sp):
        for n, (k, d) in enumerate(turns):
            print(f"  call {n}: arrays {k} dir {d} caller's stream {stream is not None}", flush=True)
            assert np.array_equal(call(k, d, stream), ref[k][d]), (n, k, d)
    bp.graph(False)
    assert np.array_equal(call(0, 0, sp), ref[0][0])
    bp.graph(True)
    assert np.array_equal(call(0, 0, sp), ref[0][0])


@pytest.mark.parametrize("N,lines,es", [(5000, 20, 8), (33000, 9, 2), (1 << 16, 5, 16),
                                        (140000, 3, 9), (3300, 40, 2)])
def test_lines_far_apart_strided(amd, N, lines, es):
    """Lines far apart with elements apart, from both entry points: as back to back, bit
    for bit; and captured in a caller's graph after a call that left the workspace too
    small for the band sums (which then go over the output), replayed several times."""
    announce(f"far lines N={N} lines={lines} es={es}")
    p = amd.FMMPlan(N, 64, 18, amd.BOTH)
    x = np.random.default_rng(N + lines).uniform(-1, 1, (lines, N))
    xs = torch.full((lines, N, es), 3.0, dtype=torch.float64, device="cuda")
    xs[:, :, 0] = torch.from_numpy(x).cuda()
    xc = xs[:, :, 0].contiguous()
    ys, yc = torch.empty_like(xs), torch.empty_like(xc)
    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    for d in (0, 1):
        p.execute_lines_device(xc.data_ptr(), yc.data_ptr(), d, lines, lines, N, 0, 1, st.cuda_stream)
        g = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        if d == 0:
            with torch.cuda.graph(g, stream=st):
                p.execute_lines_device(xs.data_ptr(), ys.data_ptr(), d, lines, lines, N * es, 0, es,
                                       torch.cuda.current_stream().cuda_stream)
            for _ in range(3):
                ys.fill_(7.0)
                g.replay()
                torch.cuda.synchronize()
                assert torch.equal(ys[:, :, 0], yc) and bool((ys[:, :, 1:] == 7.0).all())
        for fn in (amd.lib().l2c_execute_lines_device, amd.lib().l2c_execute_lines_device_noalloc):
            ys.fill_(7.0)
            torch.cuda.synchronize()
            assert fn(p.plan, xs.data_ptr(), ys.data_ptr(), d, lines, lines, N * es, 0, es,
                      st.cuda_stream) == 0
            torch.cuda.synchronize()
            assert torch.equal(ys[:, :, 0], yc) and bool((ys[:, :, 1:] == 7.0).all()), d
