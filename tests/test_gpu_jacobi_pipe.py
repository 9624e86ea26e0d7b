"""3D register-pipeline Jacobi sweeps (the default 3D path) against the CPU oracle, bit for bit, at the sizes
where a box's edges, remainders, halos and plane chunks can go wrong."""
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


# (z, y, x): the smallest; one tile of columns or rows and one more; several tiles with remainders;
# fewer planes than a pass has sweeps; rows that are not whole vectors
SHAPES_3D = [(3, 3, 3), (3, 17, 65), (4, 16, 64), (5, 25, 129), (7, 33, 121), (24, 9, 64), (23, 65, 184), (40, 40, 40),
             (64, 64, 64), (97, 31, 250), (30, 131, 333)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("bc", [0, 1])
@pytest.mark.parametrize("shape", SHAPES_3D)
def test_boxes_3d(gpu, orc, shape, bc, dtype):
    for niter, norm_every in ((1, 1), (2, 0), (13, 3), (14, 5), (22, 0)):
        _check(gpu, orc, shape, dtype, niter, bc, norm_every)


@pytest.mark.parametrize("dtype,shape", [(np.float64, (130, 257, 301)), (np.float32, (190, 251, 317)),
                                         (np.float32, (259, 300, 512))])
@pytest.mark.parametrize("bc", [0, 1])
def test_boxes_3d_tall(gpu, orc, dtype, shape, bc):
    """Fields of many boxes: the eight-row shapes, chunks of many planes."""
    _check(gpu, orc, shape, dtype, 11, bc, 6)


@pytest.mark.parametrize("bc", [0, 1])
@pytest.mark.parametrize("shape", [(80, 300, 241), (90, 260, 256)])
def test_boxes_3d_of_16_byte_lanes(gpu, orc, shape, bc):
    """FP64 in lanes of two columns, the shape of the largest fields: an odd row (whose last column is a lane's first,
    and whose last lane reaches into the next plane) and rows of whole vectors, with and without norms."""
    p = gpu.jacobi_params(shape[2], shape[1], shape[0], 22, 0, gpu.F64, bc)
    assert gpu.jacobi_route(p)["kernel"] == "register pipeline"
    for niter, norm_every in ((22, 0), (14, 5), (9, 4)):
        _check(gpu, orc, shape, np.float64, niter, bc, norm_every)
