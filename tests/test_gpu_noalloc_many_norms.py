"""cfm_jacobi_run_noalloc with so many norms that their sums fit the scratch array for fewer workgroups than a plan
launches: the kernel is chosen for those that fit, the field is the plan's bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,dtype,niter,norm_every,block", [
    # a plan's tiles here are pairs of 512 threads on each of 256 CUs; 1000 norms leave room for 256 workgroups
    ((2000, 2000), np.float64, 1000, 1, 1024), ((2000, 2001), np.float32, 3001, 3, 1024),
    ((40, 200, 200), np.float64, 5000, 5, 512), ((64, 100, 100), np.float32, 2400, 3, 512)])
@pytest.mark.parametrize("bc", [0, 1])
def test_many_norms(gpu, shape, dtype, niter, norm_every, block, bc):
    nz, ny, nx = (1,) + shape if len(shape) == 2 else shape
    init = np.random.default_rng(nx + bc).uniform(-1, 1, shape).astype(dtype)
    p = gpu.jacobi_params(nx, ny, nz, niter, norm_every, gpu.F64 if dtype == np.float64 else gpu.F32, bc)
    with gpu.DeviceBuffer.of(init) as field, gpu.DeviceBuffer(init.nbytes) as work:
        norms, t = gpu.jacobi_noalloc(p, field, work)
        out = field.download(dtype, shape)
    ref, rnorms, rt = gpu.jacobi(init, niter, bc=bc, norm_every=norm_every)
    assert np.array_equal(out, ref)
    # the same squares in other groups, each sum with its rounding kept: a few 1e-16 a group
    assert len(norms) == len(rnorms) == -(-niter // norm_every)
    assert np.allclose(norms, rnorms, rtol=1e-12, atol=0.0)
    assert t["grid_blocks"] <= (2 << 20) / 8 / len(norms) and t["block_threads"] == block
