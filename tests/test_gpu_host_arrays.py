"""Calls with host arrays: the chunked copies to the device and back (one
chunk up to 65,536 elements, then two and more, eight above 524,288), contiguous
and strided, odd lengths, in place, repeated with new data in the same arrays;
equal to the same plan on device arrays."""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 2, 255, 2001, 65536, 65537, 131072, 131073, 200001, 524289, 1000003])
@pytest.mark.parametrize("stride", [1, 3])
def test_host_equals_device(amd, N, stride):
    announce(f"host arrays N={N} stride={stride}")
    plan = amd.FMMPlan(N, 64, 18, 2)
    din, dout = amd.DeviceBuffer(N * stride), amd.DeviceBuffer(N * stride)
    buf, out = np.zeros(N * stride), np.zeros(N * stride)
    for seed in range(3):
        for d in (0, 1):
            buf[:] = np.random.default_rng(2 * seed + d).uniform(-1, 1, N * stride)
            din.upload(buf)
            dout.upload(np.full(N * stride, 7.0))
            plan.execute_device(din.ptr, dout.ptr, d, stride)
            plan.synchronize()
            out[:] = 7.0
            plan.execute(buf, d, stride, out=out)
            assert np.array_equal(out, dout.download()), (seed, d)
    if N <= 70000:
        same = buf.copy()
        plan.execute(same, 1, stride, out=same)
        assert np.array_equal(same[::stride], out[::stride])
