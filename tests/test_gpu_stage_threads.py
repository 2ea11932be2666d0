"""Host arrays on one, two, four and eight copying threads (t3x_stage.h,
threads_of): a start vector goes up and comes back after a solve of no
iterations, its bits unchanged, three times over."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1 << 20
# cells: the bytes of a vector, 24 a node, lie in this range
SHAPES = {(40, 80, 40): (2 * MB, 5 * MB), (52, 103, 52): (5 * MB, 8 * MB), (61, 121, 83): (8 * MB, 32 * MB),
          (112, 227, 112): (64 * MB, 80 * MB)}


@pytest.mark.parametrize("shape", list(SHAPES), ids=str)
def test_vector_up_and_back(shape):
    import top3d_xl_amd as t3x
    lo, hi = SHAPES[shape]
    p = t3x.Problem(np.ones(shape, bool))
    try:
        assert lo <= 24 * p.nN < hi and 24 * p.nN % (512 << 10)  # and a part of a chunk at the end
        p.set_modulus(np.ones(p.nE))
        p.assemble()
        b = p.load_vector()
        x0 = np.random.default_rng(31).standard_normal(3 * p.nN)
        x0[:3] = [np.nan, -0.0, 5e-324]
        for _ in range(3):
            x, its, _ = p.pcg(b, x0=x0, maxit=0)
            assert its == 0 and np.array_equal(x.view(np.int64), x0.view(np.int64))
            x0 = np.roll(x0, 12345)
    finally:
        p.close()
