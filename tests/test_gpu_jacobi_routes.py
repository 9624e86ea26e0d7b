"""Which kernel a Jacobi run takes, and what it says of its passes (cfm_jacobi_describe)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _route(gpu, shape, niter, norm_every=0, dtype=np.float64, bc=1, **kw):
    nz, ny, nx = (1,) + shape if len(shape) == 2 else shape
    prec = gpu.F64 if dtype == np.float64 else gpu.F32
    return gpu.jacobi_route(gpu.jacobi_params(nx, ny, nz, niter, norm_every, prec, bc, **kw))


def _pipeline_passes(niter, norm_every, bc):
    """Passes of four sweeps; one starts at each sweep whose norm is wanted, and with periodic planes the first
    sweep is one of its own."""
    k = passes = 0
    while k < niter:
        steps = min(4, niter - k)
        if norm_every:
            steps = min(steps, norm_every - k % norm_every)
        k += 1 if bc == 0 and k == 0 else steps
        passes += 1
    return passes


@pytest.mark.parametrize("bc", [0, 1])
def test_pipeline_passes(gpu, bc):
    for niter in (0, 1, 2, 3, 4, 5, 9, 40, 41, 1000):
        for norm_every in (0, 3, 4, 5, 6, 7, 10, 50, 2000):
            r = _route(gpu, (64, 64, 64), niter, norm_every, bc=bc)
            if r["kernel"] == "register pipeline":  # (norms that are too frequent go another way)
                assert r["passes"] == _pipeline_passes(niter, norm_every, bc) and r["sweeps_per_pass"] == 4
            else:
                assert niter <= 2 or norm_every == 3


def test_passes_that_are_made(gpu):
    """The benchmark's fields: a quarter of the sweeps in 3D, deeper passes in 2D."""
    assert _route(gpu, (512, 512, 512), 1000) == {"kernel": "register pipeline", "passes": 250, "sweeps_per_pass": 4}
    r = _route(gpu, (16384, 16384), 1000)
    assert r["kernel"] == "register tiles" and 4 < r["sweeps_per_pass"] <= 24
    assert r["passes"] == -(-1000 // r["sweeps_per_pass"])
    r = _route(gpu, (16384, 16384), 1000, bc=0)
    assert r["passes"] == 1 + -(-999 // r["sweeps_per_pass"])
    # one workgroup holds the field for the whole run
    assert _route(gpu, (60, 100), 777) == {"kernel": "register tiles", "passes": 1, "sweeps_per_pass": 777}


def test_passes_of_an_asked_kernel(gpu):
    assert _route(gpu, (512, 512, 512), 7, time_block=2) == {"kernel": "streaming", "passes": 4, "sweeps_per_pass": 2}
    assert _route(gpu, (512, 512, 512), 7, time_block=1)["passes"] == 7
    assert _route(gpu, (1024, 1024), 7, time_block=4)["passes"] == 2
    assert _route(gpu, (40, 40, 40), 7, variant=gpu.LAUNCH_PER_ITER)["passes"] == 7
    assert _route(gpu, (40, 40, 40), 7, variant=gpu.NO_COMPUTE)["passes"] == 0
    with pytest.raises(gpu.CfmError):
        _route(gpu, (40, 40, 2), 7)


# (shape, sweeps, norm_every, boundary) and whether the pipeline is the faster kernel there, as measured
@pytest.mark.parametrize("shape,niter,norm_every,bc,dtype,pipeline", [
    ((512, 512, 512), 40, 0, 1, np.float64, True), ((512, 512, 512), 2, 0, 1, np.float64, False),
    ((512, 512, 512), 1, 0, 1, np.float64, False), ((512, 512, 512), 4, 0, 1, np.float64, True),
    ((512, 512, 512), 4, 0, 0, np.float64, False), ((512, 512, 512), 5, 0, 0, np.float64, True),
    ((512, 512, 512), 2, 0, 0, np.float32, False), ((512, 512, 512), 40, 4, 1, np.float64, True),
    ((512, 512, 512), 40, 1, 1, np.float64, False), ((512, 512, 512), 40, 3, 1, np.float32, False),
    ((300, 300, 300), 2, 0, 0, np.float64, False), ((300, 300, 300), 3, 0, 1, np.float64, True),
    ((3, 512, 512), 2, 0, 1, np.float64, False), ((3, 512, 512), 40, 0, 1, np.float64, True),
    ((3, 512, 512), 40, 2, 1, np.float64, False), ((64, 64, 64), 1, 0, 1, np.float64, True),
    ((64, 64, 64), 40, 2, 0, np.float32, True)])
def test_pipeline_where_it_is_faster(gpu, shape, niter, norm_every, bc, dtype, pipeline):
    kernel = _route(gpu, shape, niter, norm_every, dtype, bc)["kernel"]
    assert kernel == ("register pipeline" if pipeline else "streaming")


@pytest.mark.parametrize("shape,niter,norm_every,bc,dtype,tiles", [
    ((16384, 16384), 40, 0, 1, np.float64, True), ((16384, 16384), 1, 0, 1, np.float64, False),
    ((16384, 16384), 2, 0, 1, np.float64, False), ((16384, 16384), 2, 0, 0, np.float64, False),
    ((16384, 16384), 4, 0, 0, np.float64, False), ((16384, 16384), 8, 0, 0, np.float64, True),
    ((16384, 16384), 40, 1, 1, np.float64, True), ((8192, 8192), 4, 1, 0, np.float32, False),
    ((8192, 8192), 40, 10, 0, np.float32, True), ((1024, 1024), 1, 0, 1, np.float64, True),
    ((1024, 1024), 1000, 1, 0, np.float32, True), ((5, 4000000), 40, 0, 1, np.float64, False),
    ((3, 30000000), 40, 0, 0, np.float32, False), ((32, 1000000), 40, 0, 1, np.float64, True),
    ((32, 1000000), 2, 0, 1, np.float64, False), ((3, 30000), 40, 0, 1, np.float64, True)])
def test_tiles_where_they_are_faster(gpu, shape, niter, norm_every, bc, dtype, tiles):
    kernel = _route(gpu, shape, niter, norm_every, dtype, bc)["kernel"]
    assert kernel == ("register tiles" if tiles else "streaming")


@pytest.mark.parametrize("dtype,limit", [(np.float64, 1 << 28), (np.float32, 1 << 29)])
def test_rows_of_2gib_are_no_tiles(gpu, dtype, limit):
    """(whatever the estimates say: their offsets are 32-bit)"""
    assert _route(gpu, (3, limit), 40, 0, dtype)["kernel"] == "streaming"
    assert _route(gpu, (3, limit - 4), 40, 0, dtype)["kernel"] in ("streaming", "register tiles")


# runs that keep the streaming kernels: one, two and four sweeps a pass, odd and even pass counts, x tiles, rows that
# are not whole vectors
@pytest.mark.parametrize("bc", [0, 1])
@pytest.mark.parametrize("shape,dtype,niter,norm_every", [
    ((3, 512, 512), np.float64, 2, 0), ((3, 512, 512), np.float32, 4, 1), ((3, 500, 1022), np.float64, 3, 1),
    ((3, 700, 1100), np.float32, 4, 1), ((4, 500, 515), np.float64, 2, 1), ((4, 900, 511), np.float64, 3, 1),
    ((5, 400000), np.float64, 7, 0), ((5, 400001), np.float32, 5, 2), ((6, 300002), np.float64, 4, 1),
    ((3, 1000000), np.float32, 9, 3)])
def test_streaming_by_default_bitexact(gpu, orc, shape, dtype, niter, norm_every, bc):
    assert _route(gpu, shape, niter, norm_every, dtype, bc)["kernel"] == "streaming"
    init = np.random.default_rng(shape[-1] + niter).uniform(-1, 1, shape).astype(dtype)
    ref, rnorms = orc.jacobi(init, niter, bc, norm_every)
    out, norms, _ = gpu.jacobi(init, niter, bc=bc, norm_every=norm_every)
    assert np.array_equal(out, ref)
    assert len(norms) == len(rnorms) and np.allclose(norms, rnorms, rtol=1e-10, atol=0.0)
    nz, ny, nx = (1,) + shape if len(shape) == 2 else shape
    p = gpu.jacobi_params(nx, ny, nz, niter, norm_every, gpu.F64 if dtype == np.float64 else gpu.F32, bc)
    with gpu.DeviceBuffer.of(init) as field, gpu.DeviceBuffer(init.nbytes) as work:
        nnorms, _ = gpu.jacobi_noalloc(p, field, work)
        assert np.array_equal(field.download(dtype, shape), ref) and np.array_equal(nnorms, norms)
