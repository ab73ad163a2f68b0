"""The solvers' device memory: what they keep between solves, and how it is given back."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1 << 20


def free_bytes():
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL(path).hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_kept_memory_is_bounded_and_given_back(dev, vh):
    """After a solve the library holds at most 512 MB more of the device than before, and
    vclhip_workspace_trim gives that back; the next solve gives the same x."""
    rp, col, val = vh.laplace_3d(150, 140, 130)
    n = rp.size - 1
    A, b = vh.CsrMatrix(rp, col, val), vh.DeviceArray.from_numpy(vh.random_uniform(1, n))
    x = vh.DeviceArray.zeros(n, np.float64)

    def solve():
        vh.bicgstab(A, b, x, tol=1e-6, max_iters=50)
        return x.to_numpy()

    want = solve()
    vh.workspace_trim()
    before = free_bytes()
    assert np.array_equal(solve(), want)
    kept = before - free_bytes()
    vh.workspace_trim()
    assert 0 < kept <= 512 * MB
    assert before - free_bytes() <= 2 * MB
    vh.workspace_trim()  # nothing to give back
    assert np.array_equal(solve(), want)
