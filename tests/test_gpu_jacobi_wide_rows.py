"""2D sweeps of rows of more than 2 GiB (beyond 32-bit byte offsets), on a window of columns at the rows' end."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H2D, D2H = 1, 2


@pytest.mark.parametrize("bc", [0, 1])
@pytest.mark.parametrize("dtype,limit", [(np.float64, 1 << 28), (np.float32, 1 << 29)])
def test_rows_beyond_2gib(gpu, orc, dtype, limit, bc):
    nx, ny, w, niter = limit + 70, 3, 134, 2
    size = np.dtype(dtype).itemsize
    init = np.random.default_rng(nx % 1000 + bc).uniform(-1, 1, (ny, w)).astype(dtype)
    p = gpu.jacobi_params(nx, ny, 1, niter, 0, gpu.F64 if size == 8 else gpu.F32, bc)
    hip = gpu.hip_runtime()
    at = lambda buf, row: gpu.ctypes.c_void_p(buf.ptr.value + (row * nx + nx - w) * size)
    out = np.empty_like(init)
    with gpu.DeviceBuffer(nx * ny * size) as field, gpu.DeviceBuffer(nx * ny * size) as work:
        for y in range(ny):
            assert hip.hipMemcpy(at(field, y), init[y].ctypes.data_as(gpu.ctypes.c_void_p), w * size, H2D) == 0
        gpu.jacobi_noalloc(p, field, work)
        for y in range(ny):
            assert hip.hipMemcpy(out[y].ctypes.data_as(gpu.ctypes.c_void_p), at(field, y), w * size, D2H) == 0
    ref, _ = orc.jacobi(init, niter, bc, 0)
    # (a column this close to the window's left side reads columns that the window does not hold)
    assert np.array_equal(out[:, niter + 1:], ref[:, niter + 1:])
