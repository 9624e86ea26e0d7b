"""Register-tile Jacobi sweeps (the default path of small and medium fields) against the CPU oracle, bit for
bit, at the sizes where a tile's edges, remainders and halos can go wrong."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NORM_RTOL = 1e-10  # sums of up to 1e7 squares in another order: about 1e7 * 2^-53 relative at the very most


def _check(gpu, orc, shape, dtype, niter, bc, norm_every):
    init = np.random.default_rng(sum(shape) + niter).uniform(-1, 1, shape).astype(dtype)
    out, norms, t = gpu.jacobi(init, niter, bc=bc, norm_every=norm_every)
    ref, rnorms = orc.jacobi(init, niter, bc, norm_every)
    assert np.array_equal(out, ref)
    assert len(norms) == len(rnorms) and np.allclose(norms, rnorms, rtol=NORM_RTOL, atol=0.0)


# one tile; one column or row more than a tile; several tiles with remainders of 1 and of a vector;
# rows that are not whole vectors; a field of one interior row or column
SHAPES_2D = [(3, 3), (3, 700), (700, 3), (64, 128), (64, 256), (65, 128), (64, 129), (66, 257), (97, 1031),
             (129, 130), (385, 258), (1000, 1021)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("bc", [0, 1])
@pytest.mark.parametrize("shape", SHAPES_2D)
def test_tiles_2d(gpu, orc, shape, bc, dtype):
    for niter, norm_every in ((1, 1), (2, 0), (25, 4), (53, 0)):
        _check(gpu, orc, shape, dtype, niter, bc, norm_every)


@pytest.mark.parametrize("dtype,shape", [(np.float64, (2051, 4099)), (np.float32, (2900, 7777))])
@pytest.mark.parametrize("bc", [0, 1])
def test_tiles_2d_many_rounds(gpu, orc, dtype, shape, bc):
    """More tiles than the chip holds: the two-workgroups-per-CU shapes, several tiles per workgroup."""
    _check(gpu, orc, shape, dtype, 33, bc, 16)
